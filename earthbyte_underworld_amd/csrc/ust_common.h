// Device-side helpers shared by the gfx950 kernels of the PIC Stokes hot path.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ust_kernels.h"

#define UST_BLOCK 256

#define UST_LAUNCH_CHECK()                                   \
    do {                                                     \
        hipError_t _e = hipGetLastError();                   \
        if (_e != hipSuccess) {                              \
            ust_set_hip_error(_e, __FILE__, __LINE__);       \
            return UST_EDEVICE;                              \
        }                                                    \
    } while (0)

void ust_set_hip_error(hipError_t e, const char *file, int line);
// an error message for ust_dev_error_string() from a check that is not a HIP call
void ust_set_error_text(const char *text);

static inline unsigned ust_grid_size(size_t n, unsigned block) {
    size_t g = (n + block - 1) / block;
    return (unsigned)(g == 0 ? 1 : g);
}

static inline hipStream_t ust_stream(void *s) { return (hipStream_t)s; }

// Quadratic Lagrange basis on the points {-1, 0, 1}.
__device__ __forceinline__ void lagrange3(double x, double *L) {
    L[0] = 0.5 * x * (x - 1.0);
    L[1] = 1.0 - x * x;
    L[2] = 0.5 * x * (x + 1.0);
}

// c(a, q) = 1 + s_a * xi_q for xi_q = q - 1 and s_a = 2a - 1: the factor of the Q1 shape
// function of vertex bit a evaluated at Lagrange point q (values 0, 1, 2).
__host__ __device__ constexpr int cfac(int a, int q) { return a ? q : 2 - q; }
__host__ __device__ constexpr int sgn(int a) { return 2 * a - 1; }

// Element tiles of the operator kernels: one 256-thread workgroup per tile, one element per thread.
// 2D tiles are 16 x 16 elements.  In 3D a workgroup owns a 16 x 16 column of elements and streams a chunk
// of tz element layers along z (tz from the grid size, so that a launch has enough workgroups); the K
// weights of a column are stored layer after layer, W[((txy*nz + ez)*27 + q)*256 + local], so that every
// load of a quadrature weight by a wavefront is one contiguous 64-element run, for any chunk length.  A 3D
// grid with fewer than UST_COL_MIN column layers (tnx*tny*nz) uses 16 x 4 x 4 tiles instead, stored tile
// after tile, W[(tile*27 + q)*256 + local]: small grids then get more workgroups.
#define UST_TX3 16
#define UST_TY3 16
#define UST_TTX3 16
#define UST_TTY3 4
#define UST_TTZ3 4
#define UST_TX2 16
#define UST_TY2 16
#define UST_TILE 256
#define UST_TZ3_MAX 16
#define UST_COL_MIN 1024
// workgroups a column launch aims at (the z-chunk length follows): what the GPU holds of them at two, three and four per CU
#define UST_COL_WG_TARGET 512
#define UST_COL_WG_TARGET_P 768
#define UST_COL_WG_TARGET_F32_YR 1024

struct GridDev {
    int dim;
    int col;              // 3D column layout (1) or 16x4x4 tiles (0)
    int nx, ny, nz;       // elements per axis (nz = 1 in 2D)
    int nnx, nny, nnz;    // nodes per axis
    int nel;
    int tx, ty, tz;       // tile extent in elements (3D: tz = z-chunk length of a workgroup)
    int tnx, tny, tnz;    // tiles per axis (3D: tnz = z-chunks per column)
    int ntiles;
    double hx, hy, hz;
    double sx, sy, sz;    // 2 / h per axis: no division in the kernels
    double xmin, ymin, zmin;
    double ymax;
};

// index of quadrature weight q of element (ex, ey, ez) in the tile-blocked layout
__host__ __device__ __forceinline__ size_t widx_at(const GridDev &g, int ex, int ey, int ez, int q) {
    if (g.dim == 3 && g.col) {
        const int txy = ex / UST_TX3 + g.tnx * (ey / UST_TY3);
        const int l = ex % UST_TX3 + UST_TX3 * (ey % UST_TY3);
        return (((size_t)txy * g.nz + ez) * 27 + q) * UST_TILE + l;
    }
    if (g.dim == 3) {
        const int t = ex / UST_TTX3 + g.tnx * (ey / UST_TTY3 + g.tny * (ez / UST_TTZ3));
        const int l = ex % UST_TTX3 + UST_TTX3 * (ey % UST_TTY3 + UST_TTY3 * (ez % UST_TTZ3));
        return ((size_t)t * 27 + q) * UST_TILE + l;
    }
    const int t = ex / UST_TX2 + g.tnx * (ey / UST_TY2);
    const int l = ex % UST_TX2 + UST_TX2 * (ey % UST_TY2);
    return ((size_t)t * 9 + q) * UST_TILE + l;
}

__host__ __device__ __forceinline__ size_t widx(const GridDev &g, int e, int q) {
    return widx_at(g, e % g.nx, (e / g.nx) % g.ny, e / (g.nx * g.ny), q);
}

// z-chunk of the column kernel: long enough that few node planes sit on chunk boundaries, short enough that the launch has
// about wg_target workgroups, as many as the GPU holds at once.  A few more than that leave a second round nearly empty:
// 525 workgroups at 101x67x45 took 33.7 us (FP64 product, with the gather), 420 take 29.8; 576 at 96^3 70.6 us (FP32
// prolongation pass 61.3), 504 take 55.1 (49.3); 528 at 96x64x64 37.5 us (34.2), 384 take 30.1 (27.9).  So of this and the
// longer chunks the one with the least rounds times layers is taken (and 0.7 layers for the first plane), among those
// whose workspace is no larger (for 768 workgroups: than that of 512 or of 1024).
static inline int column_chunk_least(long long columns, int nz, long long wg_target) {
    long long z = columns * nz / wg_target;
    if (z < 2) z = 2;
    if (z > UST_TZ3_MAX) z = UST_TZ3_MAX;
    return (int)(z > nz ? nz : z);
}
static inline int column_chunk(long long columns, int nz, long long wg_target) {
    const auto chunks = [&](long long z) { return (nz + z - 1) / z; };
    const auto work = [&](long long t) {
        const int z = column_chunk_least(columns, nz, t);
        return chunks(z) * (z + 1);
    };
    const auto cost = [&](long long z) { return (columns * chunks(z) + wg_target - 1) / wg_target * (10 * z + 7); };
    const long long w = work(UST_COL_WG_TARGET), v = work(UST_COL_WG_TARGET_F32_YR);
    const long long most = wg_target == UST_COL_WG_TARGET ? w : wg_target == UST_COL_WG_TARGET_F32_YR ? v : w > v ? w : v;
    int best = 0;
    for (int z = column_chunk_least(columns, nz, wg_target); z <= UST_TZ3_MAX && z <= nz; z++)
        if (chunks(z) * (z + 1) <= most && (!best || cost(z) < cost(best))) best = z;
    return best ? best : column_chunk_least(columns, nz, UST_COL_WG_TARGET);
}

// wg_target: the workgroups a column launch aims at (the z-chunk length follows)
static inline GridDev grid_dev(const ust_grid *g, long long wg_target = UST_COL_WG_TARGET) {
    GridDev d;
    d.dim = g->dim;
    d.nx = g->nel[0];
    d.ny = g->nel[1];
    d.nz = g->dim == 3 ? g->nel[2] : 1;
    d.nnx = d.nx + 1;
    d.nny = d.ny + 1;
    d.nnz = g->dim == 3 ? d.nz + 1 : 1;
    d.nel = d.nx * d.ny * d.nz;
    d.col = 0;
    if (g->dim == 3) {
        const int cnx = (d.nx + UST_TX3 - 1) / UST_TX3, cny = (d.ny + UST_TY3 - 1) / UST_TY3;
        const long long layers = (long long)cnx * cny * d.nz;
        d.col = layers >= UST_COL_MIN;
        if (d.col) {
            d.tx = UST_TX3;
            d.ty = UST_TY3;
            d.tnx = cnx;
            d.tny = cny;
            d.tz = column_chunk((long long)cnx * cny, d.nz, wg_target);
            d.tnz = (d.nz + d.tz - 1) / d.tz;
        } else {
            d.tx = UST_TTX3;
            d.ty = UST_TTY3;
            d.tz = UST_TTZ3;
            d.tnx = (d.nx + UST_TTX3 - 1) / UST_TTX3;
            d.tny = (d.ny + UST_TTY3 - 1) / UST_TTY3;
            d.tnz = (d.nz + UST_TTZ3 - 1) / UST_TTZ3;
        }
    } else {
        d.tx = UST_TX2;
        d.ty = UST_TY2;
        d.tz = 1;
        d.tnx = (d.nx + UST_TX2 - 1) / UST_TX2;
        d.tny = (d.ny + UST_TY2 - 1) / UST_TY2;
        d.tnz = 1;
    }
    d.ntiles = d.tnx * d.tny * d.tnz;
    d.hx = g->h[0];
    d.sx = 2.0 / g->h[0];
    d.sy = 2.0 / g->h[1];
    d.sz = g->dim == 3 ? 2.0 / g->h[2] : 1.0;
    d.hy = g->h[1];
    d.hz = g->dim == 3 ? g->h[2] : 1.0;
    d.xmin = g->xmin[0];
    d.ymin = g->xmin[1];
    d.zmin = g->dim == 3 ? g->xmin[2] : 0.0;
    d.ymax = g->ymax;
    return d;
}

// Workgroups go to the 8 XCDs in turn, and each XCD has its own L2.  xcd_block turns the block index into a position such
// that one XCD takes a contiguous run of positions, so tiles that share nodes and cache lines share an L2.
#define UST_XCDS 8
__device__ __forceinline__ int xcd_block(int b, int n) {
    const int x = b % UST_XCDS, q = n / UST_XCDS, r = n % UST_XCDS;
    return x * q + (x < r ? x : r) + b / UST_XCDS;
}

// Division of numbers below 2^31 by a divisor fixed for the launch, as a product (Granlund and Montgomery, "Division by
// invariant integers using multiplication"): with 2^l >= d, m = ceil(2^(31+l) / d) < 2^32 gives n / d = n m >> (31 + l).
struct FastDiv {
    unsigned d, m, s;
};
static inline FastDiv fast_div(unsigned d) {
    unsigned l = 0;
    while ((1ull << l) < d) l++;
    const unsigned long long p = 1ull << (31 + l);
    return {d, (unsigned)((p + d - 1) / d), 31 + l};
}
__device__ __forceinline__ unsigned operator/(unsigned n, const FastDiv &f) {
    return (unsigned)(((unsigned long long)n * f.m) >> f.s);
}

// position of a tile in a grid of tiles, x fastest; the division by run-time counts would be 60 scalar instructions ahead
// of a kernel's first load
struct TileDiv {
    FastDiv x, y;
};
static inline TileDiv tile_div(int nx, int ny) { return {fast_div((unsigned)nx), fast_div((unsigned)ny)}; }
__device__ __forceinline__ int3 tile_at(int tile, const TileDiv &t) {
    const unsigned r = (unsigned)tile / t.x, z = r / t.y;
    return make_int3((int)((unsigned)tile - r * t.x.d), (int)(r - z * t.y.d), (int)z);
}

// A wavefront's own LDS: its LDS operations complete in order, so a wave-level barrier (no compiler reordering across
// it) is all that one wave needs between its lanes' writes and reads of each other's values.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// bfloat16 is the upper half of an FP32: widened by a shift, narrowed with round-to-nearest-even
__device__ __forceinline__ float bf16_to_f32(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }
__device__ __forceinline__ unsigned short f32_to_bf16(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
// K weights stored as bfloat16 are read through wload<float, unsigned short>
template <typename T, typename WT>
__device__ __forceinline__ T wload(const WT *__restrict__ W, size_t i) {
    return (T)W[i];
}
template <>
__device__ __forceinline__ float wload<float, unsigned short>(const unsigned short *__restrict__ W, size_t i) {
    return bf16_to_f32(W[i]);
}
