// Discrete Voronoi cell (DVC) integration weights on gfx950.
//
// DVCWeights (PICellerator/Weights/src/DVCWeights.c): every element carries a fixed sub-grid of nx*ny(*nz)
// cells over its local box [-1,1]^dim; the particles grow their Voronoi regions over it from their seed cells,
// one particle after another, round after round, until no particle claims a cell.  A particle claims an unowned
// cell on its boundary, and takes an owned one when it is strictly nearer the cell centre than the owner
// (_ClaimCells :261-317 with _DistanceTest :604-610); its next boundary is the set of neighbours of the cells it
// has just claimed that it does not own (_UpdateBchain :395-446).  Then each particle moves to the centroid of
// its cells and weighs their volume (_GetCentroids :203-231, _Calculate3D/2D :763-925).
//
// Within one particle's turn every boundary cell is decided on its own (owner and distances only), and the next
// boundary is a set, so the reference's lists can be held in any order.  Only the particle order is sequential.
//
// k_dvc_grow: a group of G lanes owns one element, 64/G elements to a wave.  All boundary sets of an element sit
// in one ring of sub-cell indices in LDS: the particles take their turns in the same order every round, so a
// turn reads its set at the head and appends its next one at the tail.  In a turn lane t decides boundary cell t;
// the claimed cells are compacted in place, and then lane t takes neighbour t % (2 dim) of claimed cell t / (2 dim),
// with one bit per sub-cell to take each neighbour once.
// k_dvc_spill: the elements whose sets outgrew the ring (marked by a negative weight), one element to a wave with the
// sets as 64-bit words, which no element accepted by the launcher outgrows.
#include "ust_common.h"

namespace {

constexpr int DVC_LANES = 64;

struct DvcShape {
    int n[3];     // sub-grid resolution (nz = 1 in 2D)
    int ncell;    // n[0] n[1] n[2]
    int words;    // 64-bit words of a sub-cell set
    int max_np;   // particles per element the LDS layout holds
    float inv[2]; // 1 / n[0], 1 / n[1]
    int ring;     // k_dvc_grow: sub-cell indices the ring of boundary sets holds (even)
};

// floor(c / n) for 0 <= c < 4096 and 1 <= n <= 64: (c + 1/2) / n is at least 1/128 away from an integer and the
// float product errs by less than 4096 * 2^-22 < 1/1000, so the truncation is exact
__device__ __forceinline__ int small_div(int c, float inv) { return (int)(((float)c + 0.5f) * inv); }

// the (i, j, k) of sub-cell c (x fastest) without integer divisions
struct CellWalk {
    int i, j, k;
    __device__ __forceinline__ CellWalk(const DvcShape &s, int c) {
        const int t = small_div(c, s.inv[0]);
        i = c - t * s.n[0];
        k = small_div(t, s.inv[1]);
        j = t - k * s.n[1];
    }
};

// (x_o + x_p - 2 x_c).(x_o - x_p) in the reference's evaluation order, without contraction into fused
// multiply-adds: > 0 when particle p is strictly nearer the centre c than the owner o
template <int DIM>
__device__ __forceinline__ double dvc_distance_test(const double *c, const double *po, const double *pp) {
#pragma clang fp contract(off)
    double s = (po[0] + pp[0] - c[0] - c[0]) * (po[0] - pp[0]);
    s = s + (po[1] + pp[1] - c[1] - c[1]) * (po[1] - pp[1]);
    if (DIM == 3) s = s + (po[2] + pp[2] - c[2] - c[2]) * (po[2] - pp[2]);
    return s;
}

// 64-bit value of lane `src` (0 when src is outside the wave)
__device__ __forceinline__ unsigned long long lane_word(unsigned long long x, int src) {
    const int lo = __shfl((int)(unsigned)x, src & 63), hi = __shfl((int)(unsigned)(x >> 32), src & 63);
    const unsigned long long v = ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
    return (src >= 0 && src < 64) ? v : 0ull;
}

// a sub-cell set held one word per lane (lane t: sub-cells 64 t .. 64 t + 63), shifted by s sub-cells:
// bit c of up(x, s) is bit c - s of x, bit c of down(x, s) is bit c + s of x
__device__ __forceinline__ unsigned long long set_up(unsigned long long x, int s, int lane) {
    const int q = s >> 6, r = s & 63;
    const unsigned long long a = lane_word(x, lane - q);
    return r ? (a << r) | (lane_word(x, lane - q - 1) >> (64 - r)) : a;
}
__device__ __forceinline__ unsigned long long set_down(unsigned long long x, int s, int lane) {
    const int q = s >> 6, r = s & 63;
    const unsigned long long a = lane_word(x, lane + q);
    return r ? (a >> r) | (lane_word(x, lane + q + 1) << (64 - r)) : a;
}

// Region growth of one element by one wave, a boundary set as 64-bit words, word j covering sub-cells 64 j .. 64 j + 63:
// in a turn lane L decides sub-cell 64 j + L of every boundary word j that holds cells, one ballot per word, which
// leaves the claimed set one word per lane; the next boundary is that set dilated by whole-word shifts across lanes
// (+-1, +-nx, +-nx*ny sub-cells, masked at the sub-grid's x and y faces), less the cells the particle owns.
// OT: the owner grid's type, signed char when at most 127 particles share an element (less LDS, more waves)
template <int DIM, typename OT>
__device__ void dvc_element_words(const DvcShape &s, unsigned char *dvc_lds, int off, int np, double *xi0, double *xi1,
                                  double *xi2, double *w, int set_centroids, int *flag) {
    const int lane = threadIdx.x;
    const int W = s.words, ncell = s.ncell;
    // LDS: centres per axis | particle coordinates (np x DIM) | boundary sets (np x W) | owner
    double *axc = (double *)dvc_lds;                                  // n[0] + n[1] + n[2]
    double *pc = axc + (s.n[0] + s.n[1] + s.n[2]);                    // max_np * DIM
    unsigned long long *bset = (unsigned long long *)(pc + (size_t)s.max_np * DIM);  // max_np * W
    OT *owner = (OT *)(bset + (size_t)s.max_np * W);                  // ncell

    const double d[3] = {2.0 / s.n[0], 2.0 / s.n[1], 2.0 / s.n[2]};
    if (lane < DIM) {  // centres accumulated as the grid constructor does: -1 - d/2, then + d per cell
        const int n = lane == 0 ? s.n[0] : (lane == 1 ? s.n[1] : s.n[2]);
        const double dl = lane == 0 ? d[0] : (lane == 1 ? d[1] : d[2]);
        double *a = axc + (lane == 0 ? 0 : (lane == 1 ? s.n[0] : s.n[0] + s.n[1]));
        double x = -1.0 - dl / 2.0;
        for (int i = 0; i < n; i++) {
            x = x + dl;
            a[i] = x;
        }
    }
    for (int p = lane; p < np; p += DVC_LANES) {
        pc[p * DIM + 0] = xi0[off + p];
        pc[p * DIM + 1] = xi1[off + p];
        if (DIM == 3) pc[p * DIM + 2] = xi2[off + p];
    }
    for (int c = lane; c < ncell; c += DVC_LANES) owner[c] = -1;
    __syncthreads();

    const double *cxs = axc, *cys = axc + s.n[0], *czs = axc + s.n[0] + s.n[1];
    const int nx = s.n[0], nxy = s.n[0] * s.n[1];

    // per lane t < W, the sub-cells of word t that have a neighbour in -x, +x, -y, +y, and that exist
    unsigned long long m_im = 0ull, m_ip = 0ull, m_jm = 0ull, m_jp = 0ull, m_val = 0ull;
    if (lane < W) {
        CellWalk cw(s, 64 * lane);
        for (int b = 0; b < 64 && 64 * lane + b < ncell; b++) {
            const unsigned long long bit = 1ull << b;
            m_val |= bit;
            if (cw.i > 0) m_im |= bit;
            if (cw.i < nx - 1) m_ip |= bit;
            if (cw.j > 0) m_jm |= bit;
            if (cw.j < s.n[1] - 1) m_jp |= bit;
            if (++cw.i == nx) {
                cw.i = 0;
                if (++cw.j == s.n[1]) {
                    cw.j = 0;
                    cw.k++;
                }
            }
        }
    }

    // the new boundary of particle p from the set it has just claimed (lane t < W holds word t in `cw_set`;
    // owner final): the face neighbours of the claimed cells, by whole-word shifts, less the cells p owns
    auto update = [&](int p, unsigned long long cw_set) {
        unsigned long long nb = (set_up(cw_set, 1, lane) & m_im) | (set_down(cw_set, 1, lane) & m_ip) |
                                (set_up(cw_set, nx, lane) & m_jm) | (set_down(cw_set, nx, lane) & m_jp);
        if (DIM == 3) nb |= set_up(cw_set, nxy, lane) | set_down(cw_set, nxy, lane);
        nb &= m_val;
        unsigned long long live = __ballot(nb != 0ull);
        unsigned long long mine = 0ull;  // lane t < W ends with word t of the new boundary
        while (live) {
            const int j = __builtin_ctzll(live);
            live &= live - 1ull;
            const unsigned long long nj = lane_word(nb, j);
            const bool b = ((nj >> lane) & 1ull) && owner[64 * j + lane] != p;
            const unsigned long long m = __ballot(b);
            if (lane == j) mine = m;
        }
        if (lane < W) bset[(size_t)p * W + lane] = mine;
    };

    // seeds, each followed at once by its boundary (DVCWeights.c:676-696)
    for (int p = 0; p < np; p++) {
        int idx[3] = {0, 0, 0};  // every lane computes the seed (the same value)
#pragma unroll
        for (int a = 0; a < DIM; a++) {
            const double t = (pc[p * DIM + a] - (-1.0)) / d[a];
            // C truncation toward zero; k == n moves to n - 1; outside [-1, 1] (and NaN): the nearest cell
            idx[a] = (t >= 0.0) ? (t < (double)s.n[a] ? (int)t : s.n[a] - 1) : 0;
        }
        const int seed = idx[0] + idx[1] * nx + (DIM == 3 ? idx[2] * nxy : 0);
        if (lane == 0) owner[seed] = (OT)p;
        __syncthreads();
        update(p, lane == (seed >> 6) ? 1ull << (seed & 63) : 0ull);
        __syncthreads();
    }

    // rounds over the particles in order until nothing is claimed (DVCWeights.c:698-710).  Every claim changes
    // an owner and an owner only changes to a strictly nearer particle, so the rounds are bounded; the limit
    // below keeps the loop finite whatever the rounding does.
    const long long max_rounds = (long long)ncell * np + 2;
    long long rounds = 0;
    int total = 1;
    while (total != 0) {
        if (++rounds > max_rounds) {
            if (lane == 0) atomicOr(flag, 4);
            break;
        }
        total = 0;
        for (int p = 0; p < np; p++) {
            const unsigned long long *bp = bset + (size_t)p * W;
            const double *pp = pc + p * DIM;
            int claimed = 0;
            // the words of p's boundary that hold cells, one ballot; only those are visited
            const unsigned long long bmine = lane < W ? bp[lane] : 0ull;
            unsigned long long live = __ballot(bmine != 0ull);
            unsigned long long cmine = 0ull;  // lane t < W ends with word t of the claimed set
            while (live) {
                const int j = __builtin_ctzll(live);
                live &= live - 1ull;
                const unsigned long long bw = bp[j];
                const int c = 64 * j + lane;
                bool win = false;
                if ((bw >> lane) & 1ull) {
                    const int o = owner[c];
                    if (o == -1) {
                        win = true;
                    } else if (o != p) {
                        const CellWalk cw(s, c);
                        const double cc[3] = {cxs[cw.i], cys[cw.j], DIM == 3 ? czs[cw.k] : 0.0};
                        win = dvc_distance_test<DIM>(cc, pc + o * DIM, pp) > 0.0;
                    }
                    if (win) owner[c] = (OT)p;
                }
                const unsigned long long m = __ballot(win);
                if (lane == j) cmine = m;
                claimed += __popcll(m);
            }
            __syncthreads();
            update(p, cmine);
            __syncthreads();
            total += claimed;
        }
    }

    // centroids summed in sub-cell order, weight = count * cell volume (DVCWeights.c:203-231)
    const double vol = DIM == 3 ? d[0] * d[1] * d[2] : d[0] * d[1];
    for (int p = lane; p < np; p += DVC_LANES) {
        double sx = 0.0, sy = 0.0, sz = 0.0;
        int count = 0;
        int c = 0;
        for (int k = 0; k < (DIM == 3 ? s.n[2] : 1); k++)
            for (int j = 0; j < s.n[1]; j++)
                for (int i = 0; i < nx; i++, c++)
                    if (owner[c] == p) {
                        sx += cxs[i];
                        sy += cys[j];
                        if (DIM == 3) sz += czs[k];
                        count++;
                    }
        w[off + p] = (double)count * vol;
        if (set_centroids) {
            xi0[off + p] = count ? sx / count : 0.0;
            xi1[off + p] = count ? sy / count : 0.0;
            if (DIM == 3) xi2[off + p] = count ? sz / count : 0.0;
        }
    }
}

// The elements whose boundary sets outgrew k_dvc_grow's ring (it left a negative weight on their first particle): a wave
// looks at `per` elements and redoes the marked ones.  all: every element, where particles so many that k_dvc_grow's LDS
// does not fit share one.
// per: one as long as that makes few waves, since a wave redoes its elements one after the other while the GPU runs empty
// (24^3 x 100 particles with 64 to a wave 34 ms, 5.2 now; 125 on a jittered lattice, where most spill, 66 and 9.4); up to 8
// on larger swarms, where a wave without work costs more than the balance (96^3: 110,000 waves).
constexpr int DVC_SPILL_WAVES = 16384, DVC_SPILL_PER = 8;
template <int DIM, typename OT>
__global__ __launch_bounds__(DVC_LANES) void k_dvc_spill(DvcShape s, const int *cell_off, const int *elems,
                                                         int nel, double *xi0, double *xi1, double *xi2, double *w,
                                                         int set_centroids, int *flag, int per, bool all) {
    extern __shared__ __align__(16) unsigned char dvc_lds[];
    int el = blockIdx.x * per + (int)threadIdx.x;
    const bool mine = (int)threadIdx.x < per && el < nel;
    int off = 0, np = 0;
    if (mine) {
        if (elems) el = elems[el];
        off = cell_off[el];
        np = cell_off[el + 1] - off;
    }
    const bool holds = mine && np > 0 && np <= s.max_np;
    if (all && mine && !holds) atomicOr(flag, np <= 0 ? 1 : 2);
    unsigned long long todo = __ballot(holds && (all || w[off] < 0.0));
    while (todo) {
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1ull;
        dvc_element_words<DIM, OT>(s, dvc_lds, __shfl(off, j), __shfl(np, j), xi0, xi1, xi2, w, set_centroids, flag);
        __syncthreads();  // the next element reuses the LDS
    }
}

// bytes of one element's LDS in k_dvc_grow: coordinates in FP32 | ring | one bit per sub-cell | set sizes | owner
__host__ __device__ inline size_t grow_lds_element(const DvcShape &s, size_t ot) {
    return ((size_t)s.max_np * 16 + (size_t)s.ring * 2 + (size_t)((s.ncell + 31) / 32) * 4 + (size_t)s.max_np * 2 +
            (size_t)s.ncell * ot + 15) & ~(size_t)15;
}
// and of the tables all elements of a workgroup share: centres per axis | the neighbours every sub-cell has
__host__ __device__ inline size_t grow_lds_shared(const DvcShape &s) {
    return ((size_t)(s.n[0] + s.n[1] + s.n[2]) * 8 + (size_t)s.ncell + 15) & ~(size_t)15;
}

// Bound: the latency of the sequential turns (about 200 in 3D at 30 particles, some 200 VALU and 14 LDS instructions
// each), so what counts is the elements in flight, which LDS limits (40 per CU at 30 particles), and the length of a
// turn: the claim test reads FP32 coordinates in one 16-byte access, and a lane per neighbour expands five claimed
// cells a pass.  96^3 elements x 30 random particles: 151 ms with one element to a wave and the sets as words, 41 ms here
// (46 ms after an advection step, whose fullest element sizes every ring); its bytes (1.5 GB) would take 0.3 ms.
constexpr int GROW_WAVES = 2;
constexpr int DVC_WIDE_2D = 16384;  // 2D swarms of fewer elements give an element 32 lanes

template <int DIM, int G, typename OT>
__global__ __launch_bounds__(64 * GROW_WAVES) void k_dvc_grow(DvcShape s, const int *__restrict__ cell_off,
                                                              const int *__restrict__ elems, int nel, double *xi0,
                                                              double *xi1, double *xi2, double *w,
                                                              int set_centroids, int *flag) {
    static_assert(G == 16 || G == 32, "group votes are 32-bit");
    extern __shared__ __align__(16) unsigned char dvc_lds[];
    constexpr int ND = 2 * DIM;      // neighbours of a sub-cell
    constexpr int CP = G / ND;       // claimed cells expanded per pass, one lane per neighbour
    const int ncell = s.ncell, nbw = (ncell + 31) / 32;
    const unsigned R = (unsigned)s.ring;
    const int nx = s.n[0], nxy = s.n[0] * s.n[1];
    const double d[3] = {2.0 / s.n[0], 2.0 / s.n[1], 2.0 / s.n[2]};
    double *axc = (double *)dvc_lds;                                           // n[0] + n[1] + n[2]
    unsigned char *nbv = (unsigned char *)(axc + (s.n[0] + s.n[1] + s.n[2]));  // ncell: bit q = neighbour q exists
    {
        const int t = threadIdx.x;
        if (t < DIM) {  // centres accumulated as the grid constructor does: -1 - d/2, then + d per cell
            const int n = t == 0 ? s.n[0] : (t == 1 ? s.n[1] : s.n[2]);
            const double dl = t == 0 ? d[0] : (t == 1 ? d[1] : d[2]);
            double *a = axc + (t == 0 ? 0 : (t == 1 ? s.n[0] : s.n[0] + s.n[1]));
            double x = -1.0 - dl / 2.0;
            for (int i = 0; i < n; i++) {
                x = x + dl;
                a[i] = x;
            }
        }
        for (int c = t; c < ncell; c += 64 * GROW_WAVES) {
            const CellWalk q(s, c);
            nbv[c] = (unsigned char)((q.i > 0) | (q.i < nx - 1) << 1 | (q.j > 0) << 2 | (q.j < s.n[1] - 1) << 3 |
                                     (q.k > 0) << 4 | (q.k < s.n[2] - 1) << 5);
        }
    }
    const int lane = threadIdx.x & 63, gl = lane % G, grp = threadIdx.x / G;
    int e = blockIdx.x * (64 * GROW_WAVES / G) + grp;
    int off = 0, np = 0;
    if (e < nel) {
        if (elems) e = elems[e];  // the elements of a list
        off = cell_off[e];
        np = cell_off[e + 1] - off;
        if ((np <= 0 || np > s.max_np) && gl == 0) atomicOr(flag, np <= 0 ? 1 : 2);
    }
    __syncthreads();  // the tables; from here on every wave works in its own LDS
    if (np <= 0 || np > s.max_np) return;
    float4 *pf = (float4 *)(dvc_lds + grow_lds_shared(s) + grp * grow_lds_element(s, sizeof(OT)));
    unsigned short *ring = (unsigned short *)(pf + s.max_np);
    unsigned *seen = (unsigned *)(ring + R);
    unsigned short *cnt = (unsigned short *)(seen + nbw);
    OT *owner = (OT *)(cnt + s.max_np);

    // the group's lanes with pred set, and this lane's rank among them
    auto vote = [&](bool pred) -> unsigned {
        const unsigned long long b = __ballot(pred);
        if (G == 32) return lane & 32 ? (unsigned)(b >> 32) : (unsigned)b;
        return (unsigned)(b >> (lane - gl)) & 0xffffu;
    };
    const unsigned below = (1u << gl) - 1u;
    auto rank = [&](unsigned b) -> unsigned { return (unsigned)__popc(b & below); };
    auto wrap = [&](unsigned x) -> unsigned { return min(x, x - R); };  // x < 2 R: below R the difference wraps high

    // owner grid unowned, no cell seen; the particles' FP32 coordinates, and their seed cells in the set sizes' place
    for (int c = gl; c < ncell; c += G) owner[c] = -1;
    for (int c = gl; c < nbw; c += G) seen[c] = 0u;
    bool tame = true;
    for (int p = gl; p < np; p += G) {
        const double x[3] = {xi0[off + p], xi1[off + p], DIM == 3 ? xi2[off + p] : 0.0};
        int idx[3] = {0, 0, 0};
#pragma unroll
        for (int a = 0; a < DIM; a++) {
            const double t = (x[a] - (-1.0)) / d[a];
            // C truncation toward zero; k == n moves to n - 1; outside [-1, 1] (and NaN): the nearest cell
            idx[a] = (t >= 0.0) ? (t < (double)s.n[a] ? (int)t : s.n[a] - 1) : 0;
            tame = tame && fabs(x[a]) <= 1.5;
        }
        pf[p] = make_float4((float)x[0], (float)x[1], (float)x[2], 0.0f);
        cnt[p] = (unsigned short)(idx[0] + idx[1] * nx + (DIM == 3 ? idx[2] * nxy : 0));
    }
    // The claim test in FP32 first.  With |coordinates| <= 1.5 its error against the FP64 one is below 2.5e-5: centre and
    // coordinates are within 2e-7, so a factor po + pp - 2 c (at most 5) within 1.8e-6, po - pp (at most 3) within
    // 3.6e-7, each of at most three products within 8e-6.  Inside 3e-5 of zero the FP64 test decides.
    const float tol = vote(!tame) ? INFINITY : 3e-5f;
    const float fnx = (float)s.n[0], fny = (float)s.n[1];
    const float fd[3] = {(float)d[0], (float)d[1], (float)d[2]};
    const float f0[3] = {(float)(-1.0 + 0.5 * d[0]), (float)(-1.0 + 0.5 * d[1]), (float)(-1.0 + 0.5 * d[2])};
    wave_sync();

    // this lane's neighbour in the expansion of claimed cells
    const int dir = gl % ND, slot = gl / ND;
    const int step = (dir & 1 ? 1 : -1) * (dir < 2 ? 1 : (dir < 4 ? nx : nxy));
    const bool expand = gl < CP * ND;

    // seeds in particle order (a later particle seeded in the same cell takes it), each with its neighbours
    // (DVCWeights.c:676-696); none of them can be the particle's own
    unsigned head = 0, tail = 0, live = 0;
    bool spill = false;
    for (int p = 0; p < np; p++) {
        const int seed = cnt[p];
        const bool ok = gl < ND && ((nbv[seed] >> dir) & 1);
        const unsigned b = vote(ok), n = (unsigned)__popc(b);
        wave_sync();
        if (gl == 0) {
            owner[seed] = (OT)p;
            cnt[p] = (unsigned short)n;
        }
        if (ok) ring[tail + rank(b)] = (unsigned short)(seed + step);  // the ring holds more than 2 dim per particle
        tail += n;
    }
    live = tail;
    wave_sync();

    // rounds over the particles in order until every boundary is empty (DVCWeights.c:698-710).  Every claim changes an
    // owner and an owner only changes to a strictly nearer particle, so the rounds are bounded; the limit below
    // keeps the loop finite whatever the rounding does.
    const long long max_rounds = (long long)ncell * np + 2;
    long long rounds = 0;
    while (live > 0 && !spill) {
        if (++rounds > max_rounds) {
            if (gl == 0) atomicOr(flag, 4);
            break;
        }
        for (int p0 = 0; p0 < np && !spill; p0 += G) {
            unsigned turns = vote(p0 + gl < np && cnt[p0 + gl < np ? p0 + gl : 0] != 0);
            while (turns && !spill) {
                const int p = p0 + __builtin_ctz(turns);
                turns &= turns - 1u;
                const unsigned n = cnt[p];
                const float4 pp = pf[p];
                // claims, compacted in place at the head
                unsigned nc = 0;
                for (unsigned b0 = 0; b0 < n; b0 += G) {
                    bool win = false;
                    int c = 0;
                    if (b0 + gl < n) {
                        c = ring[wrap(head + b0 + gl)];
                        const int o = owner[c];
                        win = o == -1;
                        if (o >= 0 && o != p) {
                            const float4 po = pf[o];
                            // (i, j, k) as small_div takes them, in floats
                            const float fc = (float)c, ft = floorf((fc + 0.5f) * s.inv[0]);
                            const float fi = fc - ft * fnx, fk = DIM == 3 ? floorf((ft + 0.5f) * s.inv[1]) : 0.0f;
                            const float cx = f0[0] + fd[0] * fi, cy = f0[1] + fd[1] * (ft - fk * fny);
                            float t = (po.x + pp.x - 2.0f * cx) * (po.x - pp.x) + (po.y + pp.y - 2.0f * cy) * (po.y - pp.y);
                            if (DIM == 3) t += (po.z + pp.z - 2.0f * (f0[2] + fd[2] * fk)) * (po.z - pp.z);
                            win = t > tol;
                            if (!(t > tol || t < -tol)) {
                                const CellWalk cw(s, c);
                                const double cc[3] = {axc[cw.i], axc[s.n[0] + cw.j],
                                                      DIM == 3 ? axc[s.n[0] + s.n[1] + cw.k] : 0.0};
                                const double xo[3] = {xi0[off + o], xi1[off + o], DIM == 3 ? xi2[off + o] : 0.0};
                                const double xp[3] = {xi0[off + p], xi1[off + p], DIM == 3 ? xi2[off + p] : 0.0};
                                win = dvc_distance_test<DIM>(cc, xo, xp) > 0.0;
                            }
                        }
                    }
                    const unsigned b = vote(win);
                    wave_sync();
                    if (win) {
                        owner[c] = (OT)p;
                        ring[wrap(head + nc + rank(b))] = (unsigned short)c;
                    }
                    nc += (unsigned)__popc(b);
                    wave_sync();
                }
                // the neighbours of the claimed cells that p does not own, each once
                unsigned nn = 0;
                for (unsigned b0 = 0; b0 < nc; b0 += CP) {
                    bool ok = false;
                    int c1 = 0;
                    if (expand && b0 + slot < nc) {
                        const int c = ring[wrap(head + b0 + slot)];
                        c1 = c + step;
                        if (((nbv[c] >> dir) & 1) && owner[c1] != (OT)p) {
                            const unsigned bit = 1u << (c1 & 31);
                            ok = !(atomicOr(&seen[c1 >> 5], bit) & bit);
                        }
                    }
                    const unsigned b = vote(ok), m = (unsigned)__popc(b);
                    if (live + nn + m > R) {  // the claimed cells and the sets still to come stay until their turn
                        spill = true;
                        break;
                    }
                    if (ok) ring[wrap(tail + nn + rank(b))] = (unsigned short)c1;
                    nn += m;
                }
                if (spill) break;
                wave_sync();
                for (unsigned i = gl; i < nn; i += G) seen[ring[wrap(tail + i)] >> 5] = 0u;
                if (gl == 0) cnt[p] = (unsigned short)nn;
                head = wrap(head + n);
                tail = wrap(tail + nn);
                live += nn - n;
                wave_sync();
            }
        }
    }
    if (spill) {
        if (gl == 0) w[off] = -1.0;  // for k_dvc_spill, which starts from the same particles
        return;
    }

    // centroids summed in sub-cell order, weight = count * cell volume (DVCWeights.c:203-231): the owner grid turned
    // into one set of sub-cells per particle, `wc` words of 32 at a time in the ring's memory (an odd number, against
    // bank conflicts), which lane q walks for particle p0 + q
    const double vol = DIM == 3 ? d[0] * d[1] * d[2] : d[0] * d[1];
    const double *cys = axc + s.n[0], *czs = cys + s.n[1];
    unsigned *set = (unsigned *)ring;
    const int nq = np < G ? np : G;
    int wc = (int)R / 2 / nq;
    wc = wc >= nbw ? nbw | 1 : (wc - 1) | 1;
    if (wc * nq * 2 > (int)R) wc -= 2;
    for (int p0 = 0; p0 < np; p0 += G) {
        double sx = 0.0, sy = 0.0, sz = 0.0;
        int count = 0;
        for (int w0 = 0; w0 < nbw; w0 += wc) {
            const int w1 = w0 + wc < nbw ? w0 + wc : nbw, c1 = 32 * w1 < ncell ? 32 * w1 : ncell;
            for (int t = gl; t < nq * wc; t += G) set[t] = 0u;
            wave_sync();
            for (int c = 32 * w0 + gl; c < c1; c += G) {
                const int q = (int)owner[c] - p0;
                if (q >= 0 && q < nq) atomicOr(&set[q * wc + (c >> 5) - w0], 1u << (c & 31));
            }
            wave_sync();
            if (gl < nq) {
                int t = w0;
                unsigned bits = set[gl * wc];
                while (true) {
                    while (!bits && ++t < w1) bits = set[gl * wc + t - w0];
                    if (!bits) break;
                    const CellWalk cw(s, 32 * t + __builtin_ctz(bits));
                    bits &= bits - 1u;
                    count++;
                    sx += axc[cw.i];
                    sy += cys[cw.j];
                    if (DIM == 3) sz += czs[cw.k];
                }
            }
            wave_sync();
        }
        if (gl < nq && p0 + gl < np) {
            const int p = off + p0 + gl;
            w[p] = (double)count * vol;
            if (set_centroids) {
                xi0[p] = count ? sx / count : 0.0;
                xi1[p] = count ? sy / count : 0.0;
                if (DIM == 3) xi2[p] = count ? sz / count : 0.0;
            }
        }
    }
}

template <int DIM, int G, typename OT>
static int launch_dvc(const DvcShape &s, size_t lds_words, const int *cell_off, const int *elems, int nel, double *xi0,
                      double *xi1, double *xi2, double *w, int set_centroids, int *flag, hipStream_t st) {
    constexpr int EPB = 64 * GROW_WAVES / G;
    const size_t lds = grow_lds_shared(s) + EPB * grow_lds_element(s, sizeof(OT));
    const bool grow = lds <= 65536;
    if (grow)
        hipLaunchKernelGGL((k_dvc_grow<DIM, G, OT>), dim3((nel + EPB - 1) / EPB), dim3(64 * GROW_WAVES), lds, st, s,
                           cell_off, elems, nel, xi0, xi1, xi2, w, set_centroids, flag);
    const int fill = (nel + DVC_SPILL_WAVES - 1) / DVC_SPILL_WAVES;
    const int per = !grow ? 1 : fill < DVC_SPILL_PER ? fill : DVC_SPILL_PER;
    hipLaunchKernelGGL((k_dvc_spill<DIM, OT>), dim3((nel + per - 1) / per), dim3(DVC_LANES), lds_words, st, s, cell_off,
                       elems, nel, xi0, xi1, xi2, w, set_centroids, flag, per, !grow);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

}  // namespace

extern "C" {

size_t ust_k_dvc_lds_bytes(int dim, const int *res, int max_np) {
    const int nz = dim == 3 ? res[2] : 1;
    const size_t ncell = (size_t)res[0] * res[1] * nz;
    const size_t words = (ncell + 63) / 64;
    return (size_t)(res[0] + res[1] + nz) * 8 + (size_t)max_np * dim * 8 + (size_t)max_np * words * 8 +
           ncell * (max_np <= 127 ? sizeof(signed char) : sizeof(short));
}

int ust_k_dvc_weights(int dim, const int *res, int nel, const int *cell_off, int max_np, double *xi0, double *xi1,
                      double *xi2, double *w, int set_centroids, int *flag, void *stream) {
    return ust_k_dvc_weights_of(dim, res, nel, nullptr, cell_off, max_np, xi0, xi1, xi2, w, set_centroids, flag, stream);
}

int ust_k_dvc_weights_of(int dim, const int *res, int nel, const int *elems, const int *cell_off, int max_np, double *xi0,
                         double *xi1, double *xi2, double *w, int set_centroids, int *flag, void *stream) {
    if ((dim != 2 && dim != 3) || !res || nel < 0 || !cell_off || !xi0 || !xi1 || !w || !flag || max_np < 1 ||
        max_np > 32767)
        return UST_EINVAL;
    if (dim == 3 && !xi2) return UST_EINVAL;
    DvcShape s;
    s.n[0] = res[0];
    s.n[1] = res[1];
    s.n[2] = dim == 3 ? res[2] : 1;
    for (int a = 0; a < 3; a++)
        if (s.n[a] < 1 || s.n[a] > 64) return UST_EINVAL;
    s.ncell = s.n[0] * s.n[1] * s.n[2];
    if (s.ncell > 4096) return UST_EINVAL;
    s.words = (s.ncell + 63) / 64;
    s.max_np = max_np;
    s.inv[0] = 1.0f / (float)s.n[0];
    s.inv[1] = 1.0f / (float)s.n[1];
    const size_t lds = ust_k_dvc_lds_bytes(dim, res, max_np);
    if (lds > 65536) return UST_EINVAL;
    if (nel == 0) return UST_OK;
    hipStream_t st = ust_stream(stream);
    const bool narrow = max_np <= 127;
    // the ring, from the most entries that 10^dim sub-cells and random particles needed: 930 for 30 particles in 3D (1,016
    // given), 1,356 for 60 (1,406), 1,755 for 100 (1,700: a few elements spill); 123 for 20 in 2D (240).  Longer
    // rings cost waves, since LDS limits the elements in flight: 64^3 x 30 particles took 16.6 ms with 1,980 entries,
    // 14.9 ms with 1,210, 12.8 ms with 1,016.
    const int by_cell = s.ncell + 7 * max_np, by_np = 5 * s.ncell / 8 + 13 * max_np;
    s.ring = ((by_cell < by_np ? by_cell : by_np) + 1) & ~1;
#define DVC(D, G, OT) return launch_dvc<D, G, OT>(s, lds, cell_off, elems, nel, xi0, xi1, xi2, w, set_centroids, flag, st)
    // 3D boundaries hold 10 to 20 sub-cells on average: 32 lanes (64^3 x 30 particles: 12.8 ms, with 16 lanes 20.1 ms).
    // 2D ones hold 4: 16 lanes (512^2 x 20: 1.33 ms, with 32 lanes 2.05 ms), unless the elements are too few to fill
    // the GPU, where the shorter turns count (64^2 x 20: 0.126 ms with 32 lanes, 0.144 ms with 16).
    if (dim == 3 && narrow) DVC(3, 32, signed char);
    if (dim == 3) DVC(3, 32, short);
    if (nel < DVC_WIDE_2D && narrow) DVC(2, 32, signed char);
    if (nel < DVC_WIDE_2D) DVC(2, 32, short);
    if (narrow) DVC(2, 16, signed char);
    DVC(2, 16, short);
#undef DVC
}

}  // extern "C"
