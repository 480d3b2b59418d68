// PCDVC population control (PICellerator/Utils/src/PCDVC.c, non-Inflow branch) on the cell-sorted swarm.
//
// The reference walks the elements one by one, splitting particles whose discrete Voronoi region is larger than
// upperT % of the element and deleting particles whose region is smaller than lowerT %, then rebuilds the
// element's Voronoi regions.  Every element's decision depends only on its own particles, so here a group of 32 lanes
// per element counts its splits and deletions (k_pcdvc_plan), a scan turns the new counts into offsets and collects the
// elements that change (k_count_blocks, k_count_tops, k_count_offsets), and a group per element writes the new swarm
// (k_pcdvc_build).  An element that keeps its particles keeps their regions, which depend on nothing else: its weights
// and centroids are copied, and the DVC kernel runs over the changed elements alone (96^3 elements x 30 particles after an
// advection step, 15-25 % of them: 7.6-11.9 ms for 45.8).
//
// List entries of a changed element: s (original particle s of the element) or s | PCDVC_SPLIT (a copy of s at its region
// centroid).  Its list region in the scratch array starts at cell_off[e] + e * max_splits and holds at most
// n + max_splits entries.
#include "ust_common.h"

#define PCDVC_SPLIT (1 << 30)
#define PCDVC_CHANGED (1 << 30)  // in new_count: the element's particles change
constexpr int PC_LANES = 32, PC_EPB = 256 / PC_LANES;

__device__ __forceinline__ int group_sum(int v) {
    for (int off = PC_LANES / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, PC_LANES);
    return v;
}

// A thread per element read the weights uncoalesced and wrote every element's list: 634 us at 96^3 elements x 30 particles;
// a group of lanes per element, with lists for the changed ones only, 458-527 us, most of it the serial lists (2D 64x64 x
// 20: 30 -> 11 us).
// ALL: every element's list is written and the count is the count alone (ust_k_pcdvc_plan).
template <int DIM, bool ALL>
__global__ __launch_bounds__(256) void k_pcdvc_plan(GridDev g, const int *__restrict__ cell_off,
                                                    const double *__restrict__ w, const unsigned char *__restrict__ mat,
                                                    ust_pcdvc_opts o, int *__restrict__ new_count,
                                                    int *__restrict__ list, int *__restrict__ flag) {
    __shared__ int tot[3];
    if (threadIdx.x < 3) tot[threadIdx.x] = 0;
    __syncthreads();
    const int gl = threadIdx.x % PC_LANES;
    const double vol = (double)(1 << DIM);
    const double max_w = o.upper_t * vol / 100.0, min_w = o.lower_t * vol / 100.0;  // PCDVC.c:1338-1339
    for (long long e64 = (long long)blockIdx.x * PC_EPB + threadIdx.x / PC_LANES; e64 < g.nel;
         e64 += (long long)gridDim.x * PC_EPB) {
        const int e = (int)e64, p0 = cell_off[e], n = cell_off[e + 1] - p0;
        // interface element: not every particle has the first particle's material (:1160-1167)
        const int m0 = mat && n > 0 ? (int)mat[p0] : 0;
        int other = 0, big = 0, small = 0;
        for (int i = gl; i < n; i += PC_LANES) {
            const double wi = w[p0 + i];
            other |= mat && (int)mat[p0 + i] != m0;
            big += wi > max_w;
            small += wi < min_w;
        }
        const bool interface = group_sum(other) != 0;
        big = group_sum(big);
        small = group_sum(small);
        // boundary element: first or last element layer along any axis (:1171-1176)
        const int ix = e % g.nx, iy = (e / g.nx) % g.ny, iz = e / (g.nx * g.ny);
        const bool boundary = ix == 0 || ix == g.nx - 1 || iy == 0 || iy == g.ny - 1 ||
                              (DIM == 3 && (iz == 0 || iz == g.nz - 1));
        int mdel = o.max_deletions, mspl = o.max_splits;
        if (interface) {  // :1341-1345
            if (!o.delete_in_interface_cells) mdel = 0;
            if (!o.split_in_interface_cells && !boundary) mspl = 0;
        }
        if (mdel > n - 4) mdel = n / 2;  // :1373
        const int nspl = min(big, mspl), ndel = max(min(small, mdel), 0), len = n + nspl - ndel;
        const bool changed = nspl > 0 || ndel > 0;
        if (gl != 0) continue;
        new_count[e] = len | (changed && !ALL ? PCDVC_CHANGED : 0);
        if (!changed && !ALL) continue;
        int *L = list + p0 + (size_t)e * o.max_splits;
        for (int i = 0; i < n; i++) L[i] = i;
        // splits: the first mspl particles (in element order) whose region exceeds max_w (:1351, :1378-1392)
        int k = n;
        for (int i = 0; k < n + nspl; i++)
            if (w[p0 + i] > max_w) L[k++] = i | PCDVC_SPLIT;
        // deletions: candidates below min_w in decreasing swarm index; each deleted slot takes the element's last
        // entry (:1352-1359, :1404-1409; Swarm_RemoveParticleFromCell, SwarmClass.c:1055-1071)
        for (int i = n - 1; k > len; i--) {
            if (!(w[p0 + i] < min_w)) continue;
            int pos = 0;
            while (L[pos] != i) pos++;  // i is in the list: only earlier (larger) candidates were removed
            L[pos] = L[--k];
        }
        if (changed && len < 3) atomicOr(tot, 1);  // :1418-1421
        if (nspl) atomicAdd(tot + 1, nspl);
        if (ndel) atomicAdd(tot + 2, ndel);
    }
    __syncthreads();
    if (threadIdx.x == 0 && tot[0]) atomicOr(flag, 1);
    if ((threadIdx.x == 1 || threadIdx.x == 2) && tot[threadIdx.x]) atomicAdd(flag + threadIdx.x, tot[threadIdx.x]);
}

// The scan of the counts in three launches: blocks of 1024 elements, the block totals by one workgroup (which also leaves
// the totals for the host in pinned memory), the offsets.
constexpr int CNT_PER = 4, CNT_BLOCK = 256 * CNT_PER;

__device__ __forceinline__ int count_of(int c) { return c & (PCDVC_CHANGED - 1); }

// exclusive sums of v (and c) over the 256 threads, totals in *tv, *tc
template <typename T>
__device__ __forceinline__ void block_scan(T &v, int &c, T *tv, int *tc) {
    __shared__ T sv[4];
    __shared__ int sc[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T iv = v;
    int ic = c;
    for (int off = 1; off < 64; off <<= 1) {
        const T a = __shfl_up(iv, off, 64);
        const int b = __shfl_up(ic, off, 64);
        if (lane >= off) {
            iv += a;
            ic += b;
        }
    }
    __syncthreads();  // the previous use of sv, sc is over
    if (lane == 63) {
        sv[wave] = iv;
        sc[wave] = ic;
    }
    __syncthreads();
    T bv = 0;
    int bc = 0;
    *tv = 0;
    *tc = 0;
    for (int k = 0; k < 4; k++) {
        if (k < wave) {
            bv += sv[k];
            bc += sc[k];
        }
        *tv += sv[k];
        *tc += sc[k];
    }
    v = bv + iv - v;
    c = bc + ic - c;
}

// per block: particles, changed elements, the largest count, elements without particles (OFFS: cnt holds offsets)
template <bool OFFS>
__global__ __launch_bounds__(256) void k_count_blocks(const int *__restrict__ cnt, int nel, int *__restrict__ blocks,
                                                      int nb) {
    __shared__ int sm[4], se[4];
    const long long e0 = (long long)blockIdx.x * CNT_BLOCK + threadIdx.x * CNT_PER;
    int v = 0, c = 0, m = 0, z = 0;
#pragma unroll
    for (int k = 0; k < CNT_PER; k++)
        if (e0 + k < nel) {
            const int q = OFFS ? cnt[e0 + k + 1] - cnt[e0 + k] : cnt[e0 + k], len = OFFS ? q : count_of(q);
            v += len;
            c += !OFFS && (q & PCDVC_CHANGED) != 0;
            m = max(m, len);
            z += len == 0;
        }
    for (int off = 32; off > 0; off >>= 1) {
        m = max(m, __shfl_xor(m, off, 64));
        z += __shfl_xor(z, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6] = m;
        se[threadIdx.x >> 6] = z;
    }
    int tv, tc;
    block_scan(v, c, &tv, &tc);
    if (threadIdx.x == 0) {
        blocks[blockIdx.x] = tv;
        blocks[nb + blockIdx.x] = tc;
        blocks[2 * nb + blockIdx.x] = max(max(sm[0], sm[1]), max(sm[2], sm[3]));
        blocks[3 * nb + blockIdx.x] = se[0] + se[1] + se[2] + se[3];
    }
}

__global__ __launch_bounds__(256) void k_count_tops(int *__restrict__ blocks, int nb, const int *__restrict__ flag,
                                                    long long *__restrict__ host) {
    __shared__ int sm[4], se[4];
    long long base = 0;
    int cbase = 0, m = 0, z = 0;
    for (int b0 = 0; b0 < nb; b0 += 256) {
        const int b = b0 + (int)threadIdx.x;
        long long v = b < nb ? blocks[b] : 0, tv;
        int c = b < nb ? blocks[nb + b] : 0, tc;
        if (b < nb) {
            m = max(m, blocks[2 * nb + b]);
            z += blocks[3 * nb + b];
        }
        block_scan(v, c, &tv, &tc);
        if (b < nb) {
            blocks[b] = (int)(base + v);  // an overflow is refused by the host, which reads the total
            blocks[nb + b] = cbase + c;
        }
        base += tv;
        cbase += tc;
    }
    for (int off = 32; off > 0; off >>= 1) {
        m = max(m, __shfl_xor(m, off, 64));
        z += __shfl_xor(z, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6] = m;
        se[threadIdx.x >> 6] = z;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        host[0] = base;
        host[1] = cbase;
        host[2] = max(max(sm[0], sm[1]), max(sm[2], sm[3]));
        host[3] = se[0] + se[1] + se[2] + se[3];
        for (int k = 0; k < 3; k++) host[4 + k] = flag[k];
    }
}

__global__ __launch_bounds__(256) void k_count_offsets(const int *__restrict__ cnt, int nel,
                                                       const int *__restrict__ blocks, int nb, int *__restrict__ off,
                                                       int *__restrict__ elems) {
    const long long e0 = (long long)blockIdx.x * CNT_BLOCK + threadIdx.x * CNT_PER;
    int q[CNT_PER], v = 0, c = 0, tv, tc;
#pragma unroll
    for (int k = 0; k < CNT_PER; k++) {
        q[k] = e0 + k < nel ? cnt[e0 + k] : 0;
        v += count_of(q[k]);
        c += (q[k] & PCDVC_CHANGED) != 0;
    }
    block_scan(v, c, &tv, &tc);
    v += blocks[blockIdx.x];
    c += blocks[nb + blockIdx.x];
#pragma unroll
    for (int k = 0; k < CNT_PER; k++) {
        if (e0 + k >= nel) break;
        off[e0 + k] = v;
        v += count_of(q[k]);
        if (q[k] & PCDVC_CHANGED) elems[c++] = (int)(e0 + k);
        if (e0 + k + 1 == nel) off[nel] = v;
    }
}

// Bound by memory: 96^3 elements x 30 particles read and write 3.1 GB.  A thread per element, uncoalesced, took 2934 us (and
// the weights and centroids were computed again); a group of lanes per element takes 920 us, 3.4 TB/s.
// ALL: every element's particles are its list's, and only they are written (ust_k_pcdvc_build).
template <int DIM, bool ALL>
__global__ __launch_bounds__(256) void k_pcdvc_build(int nel, int max_splits, const int *__restrict__ cell_off,
                                                     const int *__restrict__ new_off, const int *__restrict__ new_count,
                                                     const int *__restrict__ list, ust_pcdvc_swarm a,
                                                     ust_pcdvc_swarm b) {
    const int gl = threadIdx.x % PC_LANES;
    for (long long e64 = (long long)blockIdx.x * PC_EPB + threadIdx.x / PC_LANES; e64 < nel;
         e64 += (long long)gridDim.x * PC_EPB) {
        const int e = (int)e64, p0 = cell_off[e], q0 = new_off[e], len = new_off[e + 1] - q0;
        const bool changed = ALL || (new_count[e] & PCDVC_CHANGED) != 0;
        const int *L = list + p0 + (size_t)e * max_splits;
        for (int k = gl; k < len; k += PC_LANES) {
            const int v = changed ? L[k] : k;
            const int src = p0 + (v & (PCDVC_SPLIT - 1)), dst = q0 + k;
            const bool split = (v & PCDVC_SPLIT) != 0;
#pragma unroll
            for (int d = 0; d < DIM; d++) {
                // a split copy takes its parent's material point and state and moves to the parent's region centroid;
                // a changed element's regions grow from its particles, the others keep theirs
                const double c = a.c[d][src], x = split ? c : a.x[d][src];
                b.x[d][dst] = x;
                if (!ALL) b.c[d][dst] = changed ? x : c;
            }
            if (!ALL) b.w[dst] = changed ? 0.0 : a.w[src];
            if (a.mat) b.mat[dst] = a.mat[src];
            if (a.coh) b.coh[dst] = a.coh[src];
            if (a.s0) b.s0[dst] = a.s0[src];
            if (a.s1) b.s1[dst] = a.s1[src];
        }
    }
}

static inline unsigned element_groups(int nel) {
    const long long b = ((long long)nel + PC_EPB - 1) / PC_EPB;
    return (unsigned)(b < 8192 ? b : 8192);
}

template <bool ALL>
static int pcdvc_plan(const ust_grid *gr, const int *cell_off, const double *w, const unsigned char *mat,
                      const ust_pcdvc_opts *o, int *new_count, int *list, int *flag, void *stream) {
    if (!gr || !cell_off || !w || !o || !new_count || !list || !flag) return UST_EINVAL;
    if (o->max_splits < 0) return UST_EINVAL;
    GridDev g = grid_dev(gr);
    if (g.nel <= 0) return UST_OK;
    if (g.dim == 3)
        hipLaunchKernelGGL((k_pcdvc_plan<3, ALL>), dim3(element_groups(g.nel)), dim3(256), 0, ust_stream(stream), g,
                           cell_off, w, mat, *o, new_count, list, flag);
    else
        hipLaunchKernelGGL((k_pcdvc_plan<2, ALL>), dim3(element_groups(g.nel)), dim3(256), 0, ust_stream(stream), g,
                           cell_off, w, mat, *o, new_count, list, flag);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_pcdvc_plan(const ust_grid *gr, const int *cell_off, const double *w, const unsigned char *mat,
                                const ust_pcdvc_opts *o, int *new_count, int *list, int *flag, void *stream) {
    return pcdvc_plan<true>(gr, cell_off, w, mat, o, new_count, list, flag, stream);
}

extern "C" int ust_k_pcdvc_plan_changed(const ust_grid *gr, const int *cell_off, const double *w, const unsigned char *mat,
                                        const ust_pcdvc_opts *o, int *new_count, int *list, int *flag, void *stream) {
    return pcdvc_plan<false>(gr, cell_off, w, mat, o, new_count, list, flag, stream);
}

extern "C" size_t ust_k_count_work_len(int nel) { return 4 * (((size_t)nel + CNT_BLOCK - 1) / CNT_BLOCK); }

static int count_blocks(int nel) { return (int)((nel + (long long)CNT_BLOCK - 1) / CNT_BLOCK); }

extern "C" int ust_k_count_offsets(int nel, const int *count, int *off, int *elems, const int *flag, long long *host,
                                   int *work, void *stream) {
    if (nel <= 0 || !count || !off || !elems || !flag || !host || !work) return UST_EINVAL;
    const int nb = count_blocks(nel);
    hipStream_t st = ust_stream(stream);
    hipLaunchKernelGGL(k_count_blocks<false>, dim3(nb), dim3(256), 0, st, count, nel, work, nb);
    hipLaunchKernelGGL(k_count_tops, dim3(1), dim3(256), 0, st, work, nb, flag, host);
    hipLaunchKernelGGL(k_count_offsets, dim3(nb), dim3(256), 0, st, count, nel, work, nb, off, elems);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_offset_stats(int nel, const int *off, const int *flag, long long *host, int *work, void *stream) {
    if (nel <= 0 || !off || !flag || !host || !work) return UST_EINVAL;
    const int nb = count_blocks(nel);
    hipStream_t st = ust_stream(stream);
    hipLaunchKernelGGL(k_count_blocks<true>, dim3(nb), dim3(256), 0, st, off, nel, work, nb);
    hipLaunchKernelGGL(k_count_tops, dim3(1), dim3(256), 0, st, work, nb, flag, host);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

template <bool ALL>
static int pcdvc_build(int dim, int nel, int max_splits, const int *cell_off, const int *new_off, const int *new_count,
                       const int *list, const ust_pcdvc_swarm &from, const ust_pcdvc_swarm &to, void *stream) {
    if (nel < 0 || max_splits < 0 || !cell_off || !new_off || !list) return UST_EINVAL;
    for (int d = 0; d < dim; d++)
        if (!from.x[d] || !from.c[d] || !to.x[d]) return UST_EINVAL;
    if ((from.mat && !to.mat) || (from.coh && !to.coh) || (from.s0 && !to.s0) || (from.s1 && !to.s1)) return UST_EINVAL;
    if (nel == 0) return UST_OK;
    if (dim == 3)
        hipLaunchKernelGGL((k_pcdvc_build<3, ALL>), dim3(element_groups(nel)), dim3(256), 0, ust_stream(stream), nel,
                           max_splits, cell_off, new_off, new_count, list, from, to);
    else
        hipLaunchKernelGGL((k_pcdvc_build<2, ALL>), dim3(element_groups(nel)), dim3(256), 0, ust_stream(stream), nel,
                           max_splits, cell_off, new_off, new_count, list, from, to);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_pcdvc_build(int dim, int nel, int max_splits, const int *cell_off, const int *new_off,
                                 const int *list, const double *xi0, const double *xi1, const double *xi2,
                                 const double *c0, const double *c1, const double *c2, const unsigned char *mat,
                                 const float *coh, const double *state0, const double *state1, double *o0, double *o1,
                                 double *o2, unsigned char *omat, float *ocoh, double *ostate0, double *ostate1,
                                 void *stream) {
    // read only
    const ust_pcdvc_swarm from = {{(double *)xi0, (double *)xi1, (double *)xi2}, {(double *)c0, (double *)c1, (double *)c2},
                                  nullptr, (unsigned char *)mat, (float *)coh, (double *)state0, (double *)state1};
    const ust_pcdvc_swarm to = {{o0, o1, o2}, {}, nullptr, omat, ocoh, ostate0, ostate1};
    return pcdvc_build<true>(dim == 3 ? 3 : 2, nel, max_splits, cell_off, new_off, nullptr, list, from, to, stream);
}

extern "C" int ust_k_pcdvc_build_changed(int dim, int nel, int max_splits, const int *cell_off, const int *new_off,
                                         const int *new_count, const int *list, const ust_pcdvc_swarm *from,
                                         const ust_pcdvc_swarm *to, void *stream) {
    if ((dim != 2 && dim != 3) || !new_count || !from || !to || !from->w || !to->w) return UST_EINVAL;
    for (int d = 0; d < dim; d++)
        if (!to->c[d]) return UST_EINVAL;
    return pcdvc_build<false>(dim, nel, max_splits, cell_off, new_off, new_count, list, *from, *to, stream);
}
