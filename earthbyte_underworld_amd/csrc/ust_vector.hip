// Krylov / smoother vector kernels (the PETSc Vec operations inside the BSSCR CG and the
// multigrid smoothers).  Scalars that the device computes (dots, CG ratios) stay in device
// memory, so a Krylov iteration issues no host round-trip except its convergence check.
#include "ust_cg.h"
#include "ust_common.h"

#define GRID_STRIDE(i, n) \
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (n); i += (size_t)gridDim.x * blockDim.x)

static inline unsigned vgrid(size_t n) {
    size_t g = (n + UST_BLOCK - 1) / UST_BLOCK;
    if (g > 8192) g = 8192;
    return (unsigned)(g == 0 ? 1 : g);
}

template <typename T>
__global__ void kv_fill(T *x, T v, size_t n) {
    GRID_STRIDE(i, n) x[i] = v;
}
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
    // splitmix64 finaliser
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
__global__ void kv_hash(double *x, size_t n, unsigned long long seed) {
    GRID_STRIDE(i, n) {
        const unsigned long long h = mix64(seed * 0x100000001B3ULL + i);
        x[i] = 2.0 * ((double)(h >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
    }
}
__global__ void kv_sign(double *x, size_t n, unsigned long long seed) {
    GRID_STRIDE(i, n) x[i] = (mix64(seed * 0x100000001B3ULL + i) >> 63) ? 1.0 : -1.0;
}
__global__ void kv_d2f(const double *x, float *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = (float)x[i];
}
__global__ void kv_d2bf(const double *x, unsigned short *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = f32_to_bf16((float)x[i]);
}
__global__ void kv_sw_step(double *pfw, const double *inc, double dt, size_t n) {
    GRID_STRIDE(i, n) {
        const double v = pfw[i] + dt * inc[i];
        pfw[i] = v < 0.0 ? 0.0 : v;
    }
}
__global__ void kv_permute(const unsigned *perm, const double *src, double *dst, size_t n) {
    GRID_STRIDE(i, n) dst[i] = src[perm[i]];
}
__global__ void kv_f2d(const float *x, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = (double)x[i];
}
__global__ void kv_axpy(double a, const double *x, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] += a * x[i];
}
__global__ void kv_axpby(double a, const double *x, double b, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = a * x[i] + b * y[i];
}
__global__ void kv_addf(const float *x, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] += (double)x[i];
}
__global__ void kv_sub(const double *a, const double *b, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = a[i] - b[i];
}
__global__ void kv_mul(const double *a, const double *b, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = a[i] * b[i];
}
__global__ void kv_div(const double *a, const double *b, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] = a[i] / b[i];
}

// two-stage deterministic reductions: stage 1 writes one partial per block (<= 1024 blocks)
template <typename TX, bool SQ, typename TY = TX>
__global__ __launch_bounds__(256) void kv_dot_stage1(const TX *x, const TY *y, size_t n, double *partial) {
    __shared__ double sh[256 / 64];
    double s = 0.0;
    GRID_STRIDE(i, n) s += SQ ? (double)x[i] * (double)y[i] : (double)x[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += sh[w];
        partial[blockIdx.x] = t;
    }
}

// sum of the stage-1 partials (one 256-thread block); the total is valid in thread 0
__device__ __forceinline__ double block_sum_partials(const double *partial, int np) {
    __shared__ double sh[4];
    double s = 0.0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) s += partial[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ __launch_bounds__(256) void kv_reduce_stage2(const double *partial, int np, double *out) {
    const double s = block_sum_partials(partial, np);
    if (threadIdx.x == 0) out[0] = s;
}

// stage 2 of r . z fused with the CG's beta, of r . r with its convergence check
__device__ __forceinline__ void cg_beta(double rz, double *rz_old, double *c) {
    if (c[1] != 0.0) return;
    c[3] = rz / rz_old[0];
    rz_old[0] = rz;
}
__device__ __forceinline__ void cg_check(double rr, double *c) {
    if (c[1] != 0.0) return;
    c[2] += 1.0;
    if (!(rr == rr)) c[1] = 2.0;
    else if (rr <= c[0]) c[1] = 1.0;
}
__global__ __launch_bounds__(256) void kv_reduce_beta(const double *partial, int np, double *rz, double *rz_old,
                                                      double *c) {
    const double s = block_sum_partials(partial, np);
    if (threadIdx.x != 0) return;
    rz[0] = s;
    cg_beta(s, rz_old, c);
}
__global__ __launch_bounds__(256) void kv_reduce_check(const double *partial, int np, double *rr, double *c) {
    const double s = block_sum_partials(partial, np);
    if (threadIdx.x != 0) return;
    rr[0] = s;
    cg_check(s, c);
}

__global__ __launch_bounds__(256) void kv_absmax_stage1(const double *x, size_t n, double *partial) {
    __shared__ double sh[4];
    double s = 0.0;
    GRID_STRIDE(i, n) s = fmax(s, fabs(x[i]));
    for (int off = 32; off > 0; off >>= 1) s = fmax(s, __shfl_xor(s, off, 64));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

__global__ __launch_bounds__(256) void kv_max_stage2(const double *partial, int np, double *out) {
    __shared__ double sh[4];
    double s = 0.0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) s = fmax(s, partial[i]);
    for (int off = 32; off > 0; off >>= 1) s = fmax(s, __shfl_xor(s, off, 64));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

static inline unsigned rgrid(size_t n) {
    size_t g = (n + UST_BLOCK * 4 - 1) / (UST_BLOCK * 4);
    if (g > 1024) g = 1024;
    return (unsigned)(g == 0 ? 1 : g);
}

__global__ void kv_mask_zero(double *x, const unsigned char *mask, size_t n) {
    GRID_STRIDE(i, n) if (mask[i]) x[i] = 0.0;
}

__global__ void kv_remove_mean(double *x, size_t n, const double *sum) {
    const double m = sum[0] / (double)n;
    GRID_STRIDE(i, n) x[i] -= m;
}

template <typename T>
__global__ void kv_cg_p(const T *z, T *p, const double *rz_new, const double *rz_old, int first, size_t n) {
    const T beta = first ? (T)0 : (T)(rz_new[0] / rz_old[0]);
    GRID_STRIDE(i, n) p[i] = z[i] + (first ? (T)0 : beta * p[i]);
}

template <typename T>
__global__ void kv_cg_xr(T *x, T *r, const T *p, const T *q, const double *num, const double *den, size_t n) {
    const T a = (T)(num[0] / den[0]);
    GRID_STRIDE(i, n) {
        x[i] += a * p[i];
        r[i] -= a * q[i];
    }
}

// The CG step by step, for callers that launch its parts themselves (the solves use the kernels of ust_cg.h), guarded by a
// control block c: c[0] threshold on r.r, c[1] state (0 running, 1 converged, 2 NaN), c[2] iterations, c[3] beta.  Once the
// state has left 0 the updates return at once.
__global__ void kv_cg_start(const double *bb, double rtol2, double *c, double *rz_old) {
    c[0] = rtol2 * bb[0];
    c[1] = bb[0] > 0.0 ? 0.0 : 1.0;
    c[2] = 0.0;
    c[3] = 0.0;
    rz_old[0] = 1.0;
}
__global__ void kv_cg_beta(const double *rz, double *rz_old, double *c) { cg_beta(rz[0], rz_old, c); }
__global__ void kv_cg_check(const double *rr, double *c) { cg_check(rr[0], c); }

template <typename TZ, typename TP>
__global__ void kv_cg_p_guarded(const TZ *z, TP *p, const double *c, size_t n) {
    if (c[1] != 0.0) return;
    const TP beta = (TP)c[3];
    GRID_STRIDE(i, n) p[i] = (TP)z[i] + beta * p[i];
}

__global__ void kv_cg_xr_guarded(double *x, double *r, const double *p, const double *q, const double *rz,
                                 const double *pq, const double *c, size_t n) {
    if (c[1] != 0.0) return;
    const double a = rz[0] / pq[0];
    GRID_STRIDE(i, n) {
        x[i] += a * p[i];
        r[i] -= a * q[i];
    }
}

// x += a p, r -= a q and the block partials of r . r (zero once converged)
template <typename T>
__global__ __launch_bounds__(256) void kv_cg_xr_rr_guarded(T *x, T *r, const T *p, const T *q, const double *rz,
                                                           const double *pq, const double *c, size_t n,
                                                           double *partial) {
    __shared__ double sh[256 / 64];
    double s = 0.0;
    if (c[1] == 0.0) {
        const T a = (T)(rz[0] / pq[0]);
        GRID_STRIDE(i, n) {
            x[i] += a * p[i];
            const T ri = r[i] - a * q[i];
            r[i] = ri;
            s += (double)ri * (double)ri;
        }
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

// y = (float)(s x)
__global__ void kv_d2f_scaled(const double *x, float *y, double s, size_t n) {
    GRID_STRIDE(i, n) y[i] = (float)(s * x[i]);
}

// The FP32 PCG's streaming kernels on 16-byte aligned vectors: four dofs per thread and step (one 16-byte load
// or store per vector), restrict-qualified so the loads of a step are issued together; the n % 4 tail dofs are
// taken by the first threads after the grid-stride loop.  The sums run in a fixed order per thread.
__device__ __forceinline__ size_t gid() { return blockIdx.x * (size_t)blockDim.x + threadIdx.x; }
__device__ __forceinline__ size_t gstride() { return (size_t)gridDim.x * blockDim.x; }

__global__ __launch_bounds__(256) void kv4_cg_xr_rr_guarded_f32(float *__restrict__ x, float *__restrict__ r,
                                                                const float *__restrict__ p,
                                                                const float *__restrict__ q, const double *rz,
                                                                const double *pq, const double *c, size_t n,
                                                                double *partial) {
    __shared__ double sh[256 / 64];
    double s = 0.0;
    if (c[1] == 0.0) {
        const float a = (float)(rz[0] / pq[0]);
        const size_t n4 = n / 4;
        float4 *x4 = (float4 *)x, *r4 = (float4 *)r;
        const float4 *p4 = (const float4 *)p, *q4 = (const float4 *)q;
        for (size_t i = gid(); i < n4; i += gstride()) {
            float4 xv = x4[i], rv = r4[i];
            const float4 pv = p4[i], qv = q4[i];
            xv.x += a * pv.x;
            xv.y += a * pv.y;
            xv.z += a * pv.z;
            xv.w += a * pv.w;
            rv.x = rv.x - a * qv.x;
            rv.y = rv.y - a * qv.y;
            rv.z = rv.z - a * qv.z;
            rv.w = rv.w - a * qv.w;
            x4[i] = xv;
            r4[i] = rv;
            s += (double)rv.x * (double)rv.x;
            s += (double)rv.y * (double)rv.y;
            s += (double)rv.z * (double)rv.z;
            s += (double)rv.w * (double)rv.w;
        }
        for (size_t i = 4 * n4 + gid(); i < n; i += gstride()) {
            x[i] += a * p[i];
            const float ri = r[i] - a * q[i];
            r[i] = ri;
            s += (double)ri * (double)ri;
        }
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ __launch_bounds__(256) void kv4_dot_f32(const float *__restrict__ x, const float *__restrict__ y, size_t n,
                                                   double *partial) {
    __shared__ double sh[256 / 64];
    double s = 0.0;
    const size_t n4 = n / 4;
    const float4 *x4 = (const float4 *)x, *y4 = (const float4 *)y;
    for (size_t i = gid(); i < n4; i += gstride()) {
        const float4 a = x4[i], b = y4[i];
        s += (double)a.x * (double)b.x;
        s += (double)a.y * (double)b.y;
        s += (double)a.z * (double)b.z;
        s += (double)a.w * (double)b.w;
    }
    for (size_t i = 4 * n4 + gid(); i < n; i += gstride()) s += (double)x[i] * (double)y[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ __launch_bounds__(256) void kv4_cg_p_guarded_f32(const float *__restrict__ z, float *__restrict__ p,
                                                            const double *c, size_t n) {
    if (c[1] != 0.0) return;
    const float beta = (float)c[3];
    const size_t n4 = n / 4;
    const float4 *z4 = (const float4 *)z;
    float4 *p4 = (float4 *)p;
    for (size_t i = gid(); i < n4; i += gstride()) {
        const float4 zv = z4[i];
        float4 pv = p4[i];
        pv.x = zv.x + beta * pv.x;
        pv.y = zv.y + beta * pv.y;
        pv.z = zv.z + beta * pv.z;
        pv.w = zv.w + beta * pv.w;
        p4[i] = pv;
    }
    for (size_t i = 4 * n4 + gid(); i < n; i += gstride()) p[i] = z[i] + beta * p[i];
}

// four consecutive values, one or two 16-byte accesses
template <typename T>
struct alignas(16) V4 {
    T v[4];
};

__device__ __forceinline__ void block_partial(double s, double *out) {
    __shared__ double sh[4];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// x = 0, r = s b (in r's type), partials of r.r, the control block
template <typename T>
__global__ __launch_bounds__(256) void kv_cg_begin(const double *__restrict__ b, double s, T *__restrict__ x,
                                                   T *__restrict__ r, size_t n, double rtol2, double *c, double *part) {
    double acc = 0.0;
    for (size_t i = gid(); i < n; i += gstride()) {
        const T v = (T)(s * b[i]);
        x[i] = (T)0;
        r[i] = v;
        acc += (double)v * (double)v;
    }
    if (blockIdx.x == 0 && threadIdx.x < 7) c[threadIdx.x] = threadIdx.x == 0 ? rtol2 : threadIdx.x == 5 ? 1.0 : 0.0;
    block_partial(acc, part + CG_RR);
}

// partials of x . y
template <typename TX, typename TY>
__global__ __launch_bounds__(256) void kv_dot_part(const TX *__restrict__ x, const TY *__restrict__ y, size_t n,
                                                   double *part) {
    double s = 0.0;
    const size_t n4 = n / 4;
    for (size_t i = gid(); i < n4; i += gstride()) {
        const V4<TX> a = ((const V4<TX> *)x)[i];
        const V4<TY> b = ((const V4<TY> *)y)[i];
#pragma unroll
        for (int k = 0; k < 4; k++) s += (double)a.v[k] * (double)b.v[k];
    }
    for (size_t i = 4 * n4 + gid(); i < n; i += gstride()) s += (double)x[i] * (double)y[i];
    block_partial(s, part);
}

// direction: p = z + (r.z / previous r.z) p, p = z in the first iteration (p is not read)
template <typename TZ, typename TP>
__global__ __launch_bounds__(256) void kv_cg_dir(const TZ *__restrict__ z, TP *__restrict__ p, double *c,
                                                 const double *part, int nrz, int nrr, size_t n) {
    const size_t n4 = n / 4;
    size_t i = gid();
    V4<TZ> zv = {};
    V4<TP> pv = {};
    if (i < n4) { /* the first vectors are on their way while the sums are formed */
        zv = ((const V4<TZ> *)z)[i];
        pv = ((const V4<TP> *)p)[i];
    }
    const CgSums s = cg_sums(part + CG_RZ, nrz, part + CG_RR, nrr, c);
    double thr = 0.0;
    const double state = cg_state(s, s.b, &thr);
    if (blockIdx.x == 0 && threadIdx.x == 0 && s.c[1] == 0.0) {
        c[1] = state;
        c[2] = s.c[4];
        c[3] = s.a;
        c[6] = thr;
    }
    if (state != 0.0) return;
    const bool first = s.c[4] == 0.0;
    const TP beta = (TP)(s.a / s.c[5]);
    while (i < n4) {
        V4<TP> o;
#pragma unroll
        for (int k = 0; k < 4; k++) o.v[k] = first ? (TP)zv.v[k] : (TP)zv.v[k] + beta * pv.v[k];
        ((V4<TP> *)p)[i] = o;
        i += gstride();
        if (i < n4) {
            zv = ((const V4<TZ> *)z)[i];
            pv = ((const V4<TP> *)p)[i];
        }
    }
    for (size_t j = 4 * n4 + gid(); j < n; j += gstride()) p[j] = first ? (TP)z[j] : (TP)z[j] + beta * p[j];
}

// step: a = r.z / p.q, x += a p, r -= a q, partials of r.r; keep: p for the next direction, where p is not its place
template <typename T>
__global__ __launch_bounds__(256) void kv_cg_step(T *__restrict__ x, T *__restrict__ r, const T *__restrict__ p,
                                                  const T *__restrict__ q, T *__restrict__ keep, double *c, double *part,
                                                  int npq, size_t n) {
    const size_t n4 = n / 4;
    size_t i = gid();
    V4<T> xv = {}, rv = {}, pv = {}, qv = {};
    if (i < n4) {
        xv = ((const V4<T> *)x)[i];
        rv = ((const V4<T> *)r)[i];
        pv = ((const V4<T> *)p)[i];
        qv = ((const V4<T> *)q)[i];
    }
    const CgSums s = cg_sums(part + CG_PQ, npq, nullptr, 0, c);
    if (s.c[1] != 0.0) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c[4] = s.c[4] + 1.0;
        c[5] = s.c[3];
    }
    const T a = (T)(s.c[3] / s.a);
    double acc = 0.0;
    while (i < n4) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            xv.v[k] += a * pv.v[k];
            rv.v[k] -= a * qv.v[k];
            acc += (double)rv.v[k] * (double)rv.v[k];
        }
        ((V4<T> *)x)[i] = xv;
        ((V4<T> *)r)[i] = rv;
        if (keep) ((V4<T> *)keep)[i] = pv;
        i += gstride();
        if (i < n4) {
            xv = ((const V4<T> *)x)[i];
            rv = ((const V4<T> *)r)[i];
            pv = ((const V4<T> *)p)[i];
            qv = ((const V4<T> *)q)[i];
        }
    }
    for (size_t j = 4 * n4 + gid(); j < n; j += gstride()) {
        x[j] += a * p[j];
        const T ri = r[j] - a * q[j];
        r[j] = ri;
        if (keep) keep[j] = p[j];
        acc += (double)ri * (double)ri;
    }
    block_partial(acc, part + CG_RR);
}

// the state after the iterations so far, for the host (pinned memory)
__global__ __launch_bounds__(256) void kv_cg_state(double *c, const double *part, int nrr, double *host) {
    const CgSums s = cg_sums(part + CG_RR, nrr, nullptr, 0, c);
    if (threadIdx.x != 0) return;
    double thr = 0.0;
    const double state = cg_state(s, s.a, &thr);
    if (s.c[1] == 0.0 && s.c[4] != 0.0) {
        c[1] = state;
        c[2] = s.c[4];
    }
    host[0] = state;
    host[1] = s.c[1] != 0.0 ? s.c[2] : s.c[4];
}

static inline bool al16(const void *a) { return ((uintptr_t)a & 15u) == 0; }

// y += s x with x in FP32: the correction of a refinement step
__global__ void kv_axpy_f32_to_f64(double s, const float *x, double *y, size_t n) {
    GRID_STRIDE(i, n) y[i] += s * (double)x[i];
}

template <typename T>
__global__ void kv_cheby(const T *b, const T *Ax, const T *invd, T *d, T *x, T c1, T c2, int first, size_t n) {
    GRID_STRIDE(i, n) {
        const T r = b[i] - Ax[i];
        const T dn = (first ? (T)0 : c1 * d[i]) + c2 * invd[i] * r;
        d[i] = dn;
        x[i] += dn;
    }
}

// first Chebyshev step from x = 0: d = c2 invd b, x = d
template <typename T>
__global__ void kv_cheby_first(const T *b, const T *invd, T *d, T *x, T c2, size_t n) {
    GRID_STRIDE(i, n) {
        const T dn = c2 * invd[i] * b[i];
        d[i] = dn;
        x[i] = dn;
    }
}

// first Chebyshev step of the FP32 V-cycle on an FP64 right-hand side: b32 = (float) b, d = c2 invd b32, x = d
__global__ void kv_cheby_first_from64(const double *b, float *b32, const float *invd, float *d, float *x, float c2,
                                      size_t n) {
    GRID_STRIDE(i, n) {
        const float bi = (float)b[i];
        const float dn = c2 * invd[i] * bi;
        b32[i] = bi;
        d[i] = dn;
        x[i] = dn;
    }
}

template <typename T>
__global__ void kv_residual(const T *b, const T *Ax, T *r, size_t n) {
    GRID_STRIDE(i, n) r[i] = b[i] - Ax[i];
}

#define LV(kern, n, ...)                                                                               \
    do {                                                                                               \
        hipLaunchKernelGGL(kern, dim3(vgrid(n)), dim3(UST_BLOCK), 0, ust_stream(stream), __VA_ARGS__); \
        UST_LAUNCH_CHECK();                                                                            \
        return UST_OK;                                                                                 \
    } while (0)

// vectors of the device-controlled CG: 16-byte aligned
template <typename... P>
static inline bool cg_vectors(size_t n, P... p) {
    return n > 0 && ((p && al16(p)) && ...);
}
template <typename TX, typename TY>
static int cg_dot(const TX *x, const TY *y, size_t n, double *part, void *stream) {
    if (!cg_vectors(n, x, y)) return UST_EINVAL;
    hipLaunchKernelGGL((kv_dot_part<TX, TY>), dim3(rgrid(n)), dim3(256), 0, ust_stream(stream), x, y, n, part);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
template <typename TZ, typename TP>
static int cg_dir(const TZ *z, TP *p, double *c, double *part, int nrz, size_t n, void *stream) {
    if (!cg_vectors(n, z, p) || nrz < 1 || nrz > UST_CG_PARTS) return UST_EINVAL;
    hipLaunchKernelGGL((kv_cg_dir<TZ, TP>), dim3(rgrid(n)), dim3(256), 0, ust_stream(stream), z, p, c, part, nrz,
                       (int)rgrid(n), n);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
template <typename T>
static int cg_step(T *x, T *r, const T *p, const T *q, T *keep, double *c, double *part, int npq, size_t n,
                   void *stream) {
    if (!cg_vectors(n, x, r, p, q) || !al16(keep) || npq < 1 || npq > UST_CG_PARTS) return UST_EINVAL;
    hipLaunchKernelGGL(kv_cg_step<T>, dim3(rgrid(n)), dim3(256), 0, ust_stream(stream), x, r, p, q, keep, c, part, npq, n);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
extern "C" {

int ust_k_fill_f64(double *x, double v, size_t n, void *stream) { LV(kv_fill<double>, n, x, v, n); }
int ust_k_fill_f32(float *x, float v, size_t n, void *stream) { LV(kv_fill<float>, n, x, v, n); }
int ust_k_fill_hash_f64(double *x, size_t n, unsigned long long seed, void *stream) {
    LV(kv_hash, n, x, n, seed);
}
int ust_k_fill_sign_f64(double *x, size_t n, unsigned long long seed, void *stream) {
    LV(kv_sign, n, x, n, seed);
}
int ust_k_copy_f64_to_f32(const double *x, float *y, size_t n, void *stream) { LV(kv_d2f, n, x, y, n); }
int ust_k_copy_f32_to_f64(const float *x, double *y, size_t n, void *stream) { LV(kv_f2d, n, x, y, n); }
int ust_k_copy_f64_to_bf16(const double *x, unsigned short *y, size_t n, void *stream) { LV(kv_d2bf, n, x, y, n); }
int ust_k_strain_weakening_step(double *pfw, const double *pfw_inc, int np, double dt, void *stream) {
    if (np < 0 || (np > 0 && (!pfw || !pfw_inc))) return UST_EINVAL;
    LV(kv_sw_step, (size_t)np, pfw, pfw_inc, dt, (size_t)np);
}
int ust_k_permute_f64(const unsigned *perm, const double *src, double *dst, int n, void *stream) {
    if (n < 0 || (n > 0 && (!perm || !src || !dst))) return UST_EINVAL;
    LV(kv_permute, (size_t)n, perm, src, dst, (size_t)n);
}
int ust_k_axpy_f64(double a, const double *x, double *y, size_t n, void *stream) { LV(kv_axpy, n, a, x, y, n); }
int ust_k_axpby_f64(double a, const double *x, double b, double *y, size_t n, void *stream) {
    LV(kv_axpby, n, a, x, b, y, n);
}
int ust_k_add_f32_to_f64(const float *x, double *y, size_t n, void *stream) { LV(kv_addf, n, x, y, n); }
int ust_k_sub_f64(const double *a, const double *b, double *y, size_t n, void *stream) { LV(kv_sub, n, a, b, y, n); }
int ust_k_scale_mul_f64(const double *a, const double *b, double *y, size_t n, void *stream) {
    LV(kv_mul, n, a, b, y, n);
}
int ust_k_div_f64(const double *a, const double *b, double *y, size_t n, void *stream) { LV(kv_div, n, a, b, y, n); }

int ust_k_dot_f64(const double *x, const double *y, size_t n, double *partial, double *out, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL((kv_dot_stage1<double, true>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_stage2, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, out);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

int ust_k_dot_f32(const float *x, const float *y, size_t n, double *partial, double *out, void *stream) {
    const unsigned g = rgrid(n);
    if (al16(x) && al16(y))
        hipLaunchKernelGGL(kv4_dot_f32, dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    else
        hipLaunchKernelGGL((kv_dot_stage1<float, true>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_stage2, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, out);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

int ust_k_sum_f64(const double *x, size_t n, double *partial, double *out, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL((kv_dot_stage1<double, false>), dim3(g), dim3(256), 0, ust_stream(stream), x, x, n, partial);
    hipLaunchKernelGGL(kv_reduce_stage2, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, out);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

int ust_k_absmax_f64(const double *x, size_t n, double *partial, double *out, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL(kv_absmax_stage1, dim3(g), dim3(256), 0, ust_stream(stream), x, n, partial);
    hipLaunchKernelGGL(kv_max_stage2, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, out);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

int ust_k_mask_zero_f64(double *x, const unsigned char *mask, size_t n, void *stream) {
    LV(kv_mask_zero, n, x, mask, n);
}

int ust_k_remove_mean_f64(double *x, size_t n, const double *sum, void *stream) {
    LV(kv_remove_mean, n, x, n, sum);
}

int ust_k_cg_update_p_f64(const double *z, double *p, const double *rz_new, const double *rz_old, int first, size_t n,
                          void *stream) {
    LV(kv_cg_p<double>, n, z, p, rz_new, rz_old, first, n);
}
int ust_k_cg_update_p_f32(const float *z, float *p, const double *rz_new, const double *rz_old, int first, size_t n,
                          void *stream) {
    LV(kv_cg_p<float>, n, z, p, rz_new, rz_old, first, n);
}
int ust_k_cg_update_xr_f64(double *x, double *r, const double *p, const double *q, const double *num,
                           const double *den, size_t n, void *stream) {
    LV(kv_cg_xr<double>, n, x, r, p, q, num, den, n);
}
int ust_k_cg_update_xr_f32(float *x, float *r, const float *p, const float *q, const double *num, const double *den,
                           size_t n, void *stream) {
    LV(kv_cg_xr<float>, n, x, r, p, q, num, den, n);
}

int ust_k_cg_parts(size_t n) { return (int)rgrid(n); }
int ust_k_cg_begin_f64(const double *b, double *x, double *r, size_t n, double rtol2, double *c, double *part,
                       void *stream) {
    if (!cg_vectors(n, b, x, r)) return UST_EINVAL;
    hipLaunchKernelGGL(kv_cg_begin<double>, dim3(rgrid(n)), dim3(256), 0, ust_stream(stream), b, 1.0, x, r, n, rtol2, c,
                       part);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_cg_begin_f32(const double *b, double s, float *x, float *r, size_t n, double rtol2, double *c, double *part,
                       void *stream) {
    if (!cg_vectors(n, b, x, r)) return UST_EINVAL;
    hipLaunchKernelGGL(kv_cg_begin<float>, dim3(rgrid(n)), dim3(256), 0, ust_stream(stream), b, s, x, r, n, rtol2, c,
                       part);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_cg_dot_rz_f64(const double *r, const double *z, size_t n, double *part, void *stream) {
    return cg_dot(r, z, n, part + CG_RZ, stream);
}
int ust_k_cg_dot_rz_zf(const double *r, const float *z, size_t n, double *part, void *stream) {
    return cg_dot(r, z, n, part + CG_RZ, stream);
}
int ust_k_cg_dot_rz_f32(const float *r, const float *z, size_t n, double *part, void *stream) {
    return cg_dot(r, z, n, part + CG_RZ, stream);
}
int ust_k_cg_dot_pq_f64(const double *p, const double *q, size_t n, double *part, void *stream) {
    return cg_dot(p, q, n, part + CG_PQ, stream);
}
int ust_k_cg_dot_pq_f32(const float *p, const float *q, size_t n, double *part, void *stream) {
    return cg_dot(p, q, n, part + CG_PQ, stream);
}
int ust_k_cg_dir_f64(const double *z, double *p, double *c, double *part, int nrz, size_t n, void *stream) {
    return cg_dir(z, p, c, part, nrz, n, stream);
}
int ust_k_cg_dir_zf(const float *z, double *p, double *c, double *part, int nrz, size_t n, void *stream) {
    return cg_dir(z, p, c, part, nrz, n, stream);
}
int ust_k_cg_dir_f32(const float *z, float *p, double *c, double *part, int nrz, size_t n, void *stream) {
    return cg_dir(z, p, c, part, nrz, n, stream);
}
int ust_k_cg_step_f64(double *x, double *r, const double *p, const double *q, double *keep, double *c, double *part, int npq,
                      size_t n, void *stream) {
    return cg_step(x, r, p, q, keep, c, part, npq, n, stream);
}
int ust_k_cg_step_f32(float *x, float *r, const float *p, const float *q, float *keep, double *c, double *part, int npq,
                      size_t n, void *stream) {
    return cg_step(x, r, p, q, keep, c, part, npq, n, stream);
}
int ust_k_cg_state(double *c, const double *part, size_t n, double *host, void *stream) {
    hipLaunchKernelGGL(kv_cg_state, dim3(1), dim3(256), 0, ust_stream(stream), c, part, (int)rgrid(n), host);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

int ust_k_cheby_first_from_f64(const double *b, float *b32, const float *invd, float *d, float *x, float c2,
                               size_t n, void *stream) {
    LV(kv_cheby_first_from64, n, b, b32, invd, d, x, c2, n);
}
int ust_k_cg_start(const double *bb, double rtol2, double *ctl, double *rz_old, void *stream) {
    hipLaunchKernelGGL(kv_cg_start, dim3(1), dim3(1), 0, ust_stream(stream), bb, rtol2, ctl, rz_old);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_cg_beta(const double *rz, double *rz_old, double *ctl, void *stream) {
    hipLaunchKernelGGL(kv_cg_beta, dim3(1), dim3(1), 0, ust_stream(stream), rz, rz_old, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_cg_check(const double *rr, double *ctl, void *stream) {
    hipLaunchKernelGGL(kv_cg_check, dim3(1), dim3(1), 0, ust_stream(stream), rr, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_cg_p_guarded_f64(const double *z, double *p, const double *ctl, size_t n, void *stream) {
    LV((kv_cg_p_guarded<double, double>), n, z, p, ctl, n);
}
int ust_k_cg_p_guarded_zf(const float *z, double *p, const double *ctl, size_t n, void *stream) {
    LV((kv_cg_p_guarded<float, double>), n, z, p, ctl, n);
}
int ust_k_cg_xr_guarded_f64(double *x, double *r, const double *p, const double *q, const double *rz,
                            const double *pq, const double *ctl, size_t n, void *stream) {
    LV(kv_cg_xr_guarded, n, x, r, p, q, rz, pq, ctl, n);
}
int ust_k_cg_xr_rr_guarded_f64(double *x, double *r, const double *p, const double *q, const double *rz,
                               const double *pq, double *ctl, size_t n, double *partial, double *rr,
                               void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL(kv_cg_xr_rr_guarded<double>, dim3(g), dim3(256), 0, ust_stream(stream), x, r, p, q, rz, pq, ctl, n,
                       partial);
    hipLaunchKernelGGL(kv_reduce_check, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, rr, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_dot_mixed(const double *x, const float *y, size_t n, double *partial, double *out, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL((kv_dot_stage1<double, true, float>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_stage2, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, out);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_dot_mixed_beta(const double *x, const float *y, size_t n, double *partial, double *rz, double *rz_old,
                         double *ctl, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL((kv_dot_stage1<double, true, float>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_beta, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, rz, rz_old, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_dot_beta_f64(const double *x, const double *y, size_t n, double *partial, double *rz, double *rz_old,
                       double *ctl, void *stream) {
    const unsigned g = rgrid(n);
    hipLaunchKernelGGL((kv_dot_stage1<double, true>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_beta, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, rz, rz_old, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_dot_beta_f32(const float *x, const float *y, size_t n, double *partial, double *rz, double *rz_old,
                       double *ctl, void *stream) {
    const unsigned g = rgrid(n);
    if (al16(x) && al16(y))
        hipLaunchKernelGGL(kv4_dot_f32, dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    else
        hipLaunchKernelGGL((kv_dot_stage1<float, true>), dim3(g), dim3(256), 0, ust_stream(stream), x, y, n, partial);
    hipLaunchKernelGGL(kv_reduce_beta, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, rz, rz_old, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_copy_f64_to_f32_scaled(const double *x, float *y, double s, size_t n, void *stream) {
    LV(kv_d2f_scaled, n, x, y, s, n);
}
int ust_k_cg_p_guarded_f32(const float *z, float *p, const double *ctl, size_t n, void *stream) {
    if (al16(z) && al16(p)) LV(kv4_cg_p_guarded_f32, (n + 3) / 4, z, p, ctl, n);
    LV((kv_cg_p_guarded<float, float>), n, z, p, ctl, n);
}
int ust_k_cg_xr_rr_guarded_f32(float *x, float *r, const float *p, const float *q, const double *rz, const double *pq,
                               double *ctl, size_t n, double *partial, double *rr, void *stream) {
    const unsigned g = rgrid(n);
    if (al16(x) && al16(r) && al16(p) && al16(q))
        hipLaunchKernelGGL(kv4_cg_xr_rr_guarded_f32, dim3(g), dim3(256), 0, ust_stream(stream), x, r, p, q, rz, pq, ctl,
                           n, partial);
    else
        hipLaunchKernelGGL(kv_cg_xr_rr_guarded<float>, dim3(g), dim3(256), 0, ust_stream(stream), x, r, p, q, rz, pq, ctl,
                           n, partial);
    hipLaunchKernelGGL(kv_reduce_check, dim3(1), dim3(256), 0, ust_stream(stream), partial, (int)g, rr, ctl);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
int ust_k_axpy_f32_to_f64(double s, const float *x, double *y, size_t n, void *stream) {
    LV(kv_axpy_f32_to_f64, n, s, x, y, n);
}
int ust_k_cheby_step_f64(const double *b, const double *Ax, const double *invd, double *d, double *x, double c1,
                         double c2, size_t n, void *stream) {
    LV(kv_cheby<double>, n, b, Ax, invd, d, x, c1, c2, c1 == 0.0 ? 1 : 0, n);
}
int ust_k_cheby_step_f32(const float *b, const float *Ax, const float *invd, float *d, float *x, float c1, float c2,
                         size_t n, void *stream) {
    LV(kv_cheby<float>, n, b, Ax, invd, d, x, c1, c2, c1 == 0.0f ? 1 : 0, n);
}
int ust_k_cheby_first_f64(const double *b, const double *invd, double *d, double *x, double c2, size_t n,
                          void *stream) {
    LV(kv_cheby_first<double>, n, b, invd, d, x, c2, n);
}
int ust_k_cheby_first_f32(const float *b, const float *invd, float *d, float *x, float c2, size_t n, void *stream) {
    LV(kv_cheby_first<float>, n, b, invd, d, x, c2, n);
}
int ust_k_residual_f64(const double *b, const double *Ax, double *r, size_t n, void *stream) {
    LV(kv_residual<double>, n, b, Ax, r, n);
}
int ust_k_residual_f32(const float *b, const float *Ax, float *r, size_t n, void *stream) {
    LV(kv_residual<float>, n, b, Ax, r, n);
}

}  // extern "C"
