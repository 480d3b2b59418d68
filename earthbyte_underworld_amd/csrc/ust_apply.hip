// The hot operator of the BSSCR solve on gfx950: y = K u, matrix-free, from the 3^dim quadrature
// weights of each element (the MatMult of the A11 block, auglag-driver-DGTGD.c:191-403, that every
// inner Krylov iteration and every multigrid smoothing step performs, PETScMGSolver.c:641-716).
//
// 3D: one 256-thread workgroup owns a 16x16 column of elements, one element per thread, and streams a
// chunk of element layers along z.  Node planes are staged in LDS once each; per layer every thread applies
// its element (element_apply3 below, about 600 operations) and leaves its 8 vertex results in LDS; each node
// of the plane below the layer then sums, in a fixed order, the contributions of the (up to) four elements
// above it and the four below it (carried in registers from the previous layer), and is finished: written to
// y through the epilogue, unless it lies on the ring of the column (shared with a neighbouring column) or on
// a chunk-boundary plane (shared with the next chunk).  Those nodes go to the workgroup's slot of a workspace,
// and a second, node-ordered pass sums the two to eight slots covering each of them.  No atomics touch memory
// and the summation order is fixed, so K u is bitwise reproducible.
// Grids with fewer than 1024 column layers (the coarse multigrid levels) use 16x4x4 tiles instead, one per
// workgroup, which gives small grids more workgroups, and the smaller of those (halo_grid below) and all 2D grids the halo
// kernels: a workgroup owns a block of nodes and computes every element that touches it, without a workspace.  Passes that
// overwrite what neighbouring workgroups stage take tiles there too (2D: 16x16 elements, the same workspace scheme).
#include <mutex>
#include <stdio.h>

#include "ust_cg.h"
#include "ust_common.h"

// axes orthogonal to k, in increasing order
__host__ __device__ constexpr int P1(int k) { return k == 0 ? 1 : 0; }
__host__ __device__ constexpr int P2(int k) { return k == 2 ? 1 : 2; }
__host__ __device__ constexpr int pow3(int k) { return k == 0 ? 1 : (k == 1 ? 3 : 9); }

// ------------------------------------------------------------------------------------------
// Element action y = K_e u in 3D, in edge differences.  A velocity component is trilinear, so d u_i / d x_k is constant
// along k and, over the other two axes, interpolates the differences of u_i along the element's four edges in direction
// k with products of hat functions; the test functions' gradients are the same.  The weights W at {-1,0,1}^3 therefore
// enter through their sums against products of two hats per axis -- N0 N0, N0 N1, N1 N1, at a line of three weights
// W0 + W1 / 4, W1 / 4, W2 + W1 / 4, or against one hat or none where only one or none varies along it:
//   S_k  (9, per direction k): the 4 x 4 products of the differences along k with themselves, one component at a time,
//   L_ik (12, per pair): the 4 x 4 products of the differences of u_i along k with those of u_k along i.
// Per element 120 operations for S (four times) and 114 for L, 36 differences, 240 multiply-adds, 24 scalings and 72 to the
// vertices: 606.  Interpolating gradients to and stresses from the 27 points takes about 750; monomials around the
// element's centre, whose products share terms, 456.  But those round sums and differences of all eight vertices on the
// way in and out, each vertex's result by the element's largest, where here a difference is rounded once before it is
// used and, of weights of one sign, every sum is of one sign.  Error of the product of a random field, relative 2-norm,
// and time at 128x128x64 with the gather -- points: FP32 5.39e-8, FP64 1.57e-16, 49.0 and 86.6 us; monomials: 6.45e-8,
// 1.68e-16, 38.4 and 67.1 us; edges: 5.35e-8, 1.55e-16, 42.3 and 71.1 us.  Other grids: FP32 101x67x45 5.49, 6.73, 5.34e-8;
// 60x44x40 (tiles) 4.87, 6.10, 4.85e-8; 64x64x32, where powers of two scale the points without rounding, 4.70, 5.83,
// 4.91e-8; FP64 40x36x30 (halo) 1.69, 1.88, 1.57e-16.
// ------------------------------------------------------------------------------------------
// lower end of edge b in direction k: bit 0 of b on axis P1(k), bit 1 on P2(k)
__host__ __device__ constexpr int edge3(int k, int b) { return (b & 1) << P1(k) | (b >> 1) << P2(k); }
// the edge of direction k at bits (bi, bj) of the axes i and j
__host__ __device__ constexpr int edge_at(int k, int i, int bi, int bj) { return P1(k) == i ? bi | bj << 1 : bj | bi << 1; }

// factors of the gradients' products: w[k] = (1 / (4 h_k))^2 and r[i][k] = h_k / h_i
template <typename T>
struct GradScale {
    T w[3], r[3][3];
};
template <typename T>
static inline GradScale<T> grad_scale(const GridDev &g) {
    const double d[3] = {g.sx, g.sy, g.sz};  // 2 / h
    GradScale<T> s;
    for (int k = 0; k < 3; k++) {
        s.w[k] = (T)(0.125 * d[k] * (0.125 * d[k]));
        for (int i = 0; i < 3; i++) s.r[i][k] = (T)(d[i] / d[k]);
    }
    return s;
}

template <typename T, int I, int K, typename U>
__device__ __forceinline__ void differences3(const U &u, T d[4]) {
#pragma unroll
    for (int b = 0; b < 4; b++) d[b] = u(edge3(K, b) | 1 << K, I) - u(edge3(K, b), I);
}

// 16 S_K, index q1 + 3 q2 with q the number of upper hats on P1(K) and P2(K)
template <typename T, int K>
__device__ __forceinline__ void edge_weights3(const T W[27], T S[9]) {
    constexpr int k = pow3(K), p = pow3(P1(K)), q = pow3(P2(K));
#pragma unroll
    for (int j = 0; j < 3; j++) {
        T l[3];
#pragma unroll
        for (int i = 0; i < 3; i++) l[i] = (W[i * p + j * q] + W[i * p + j * q + 2 * k]) + W[i * p + j * q + k];
        S[3 * j] = (T)4 * l[0] + l[1];
        S[3 * j + 1] = l[1];
        S[3 * j + 2] = (T)4 * l[2] + l[1];
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        S[i] = (T)4 * S[i] + S[3 + i];
        S[6 + i] = (T)4 * S[6 + i] + S[3 + i];
    }
}

// 16 L_IK: one hat on I (first index) and on K, two on the third axis (last index: the number of upper ones)
template <typename T, int I, int K>
__device__ __forceinline__ void cross_weights3(const T W[27], T L[2][2][3]) {
    constexpr int i = pow3(I), k = pow3(K), j = pow3(3 - I - K);
#pragma unroll
    for (int a = 0; a < 2; a++) {
        T m[3][3];
#pragma unroll
        for (int n = 0; n < 9; n++) {
            const int o = (n % 3) * k + (n / 3) * j;
            m[n % 3][n / 3] = (T)2 * W[o + 2 * a * i] + W[o + i];
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            T l[3];
#pragma unroll
            for (int n = 0; n < 3; n++) l[n] = (T)2 * m[2 * b][n] + m[1][n];
            L[a][b][0] = (T)4 * l[0] + l[1];
            L[a][b][1] = l[1];
            L[a][b][2] = (T)4 * l[2] + l[1];
        }
    }
}

// r += S d, the product with the largest weight last
template <typename T>
__device__ __forceinline__ void edge_product3(const T S[9], const T d[4], T r[4]) {
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int n = 1; n < 5; n++) {
            const int b = a ^ (n & 3);
            r[a] += S[(a & 1) + (b & 1) + 3 * ((a >> 1) + (b >> 1))] * d[b];
        }
}

// the edges' w r to the vertices
template <typename T, int I, int K, bool FIRST>
__device__ __forceinline__ void edges_to_vertices3(const T r[4], T w, T y[8][3]) {
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int a = edge3(K, b);
        y[a | 1 << K][I] = FIRST ? w * r[b] : y[a | 1 << K][I] + w * r[b];
        y[a][I] = FIRST ? -(w * r[b]) : y[a][I] - w * r[b];
    }
}

// between the parts of an element's action, kept APART: instructions of one are not moved among those of another.
// Interleaved, several parts' sums are held at once: the FP64 column kernel (256 registers) then spills 10 of them, the FP32
// product's (128) 12.  The kernels of small grids have registers to spare and hide the latency of one part behind another:
// 24x16x16 FP64 product 5.1 us, with the parts apart 5.6; 64x64x32 (tiles) 13.2, 13.6.
template <bool APART>
__device__ __forceinline__ void part_end() {
    if (APART) __builtin_amdgcn_sched_barrier(0);
}

// d u_I / d x_K with itself (S_K) and with d u_K / d x_I (L_IK), and the same with I and K exchanged.  SI, SK: the edge
// weights, made here (NEW) or by a part before
template <bool APART, typename T, int I, int K, bool FIRST_I, bool FIRST_K, bool NEW_I, bool NEW_K, typename U>
__device__ __forceinline__ void pair3(const U &u, const T W[27], T SI[9], T SK[9], const GradScale<T> &s, T y[8][3]) {
    T di[4], dk[4], ri[4], rk[4];
    {
        T L[2][2][3];
        cross_weights3<T, I, K>(W, L);
        differences3<T, I, K>(u, di);
        differences3<T, K, I>(u, dk);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                T vi = (T)0, vk = (T)0;
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    const int b = n & 1, e = n >> 1;
                    vi += L[a][b][c + e] * dk[edge_at(I, K, b, e)];
                    vk += L[b][a][c + e] * di[edge_at(K, I, b, e)];
                }
                ri[edge_at(K, I, a, c)] = s.r[I][K] * vi;
                rk[edge_at(I, K, a, c)] = s.r[K][I] * vk;
            }
    }
    part_end<APART>();
    if (NEW_K) edge_weights3<T, K>(W, SK);
    edge_product3<T>(SK, di, ri);
    edges_to_vertices3<T, I, K, FIRST_I>(ri, s.w[K], y);
    part_end<APART>();
    if (NEW_I) edge_weights3<T, I>(W, SI);
    edge_product3<T>(SI, dk, rk);
    edges_to_vertices3<T, K, I, FIRST_K>(rk, s.w[I], y);
    part_end<APART>();
}

// d u_K / d x_K with itself, which its strain holds twice
template <bool APART, typename T, int K, typename U>
__device__ __forceinline__ void normal3(const U &u, const T S[9], const GradScale<T> &s, T y[8][3]) {
    T d[4], r[4] = {(T)0, (T)0, (T)0, (T)0};
    differences3<T, K, K>(u, d);
    edge_product3<T>(S, d, r);
    edges_to_vertices3<T, K, K, false>(r, (T)2 * s.w[K], y);
    part_end<APART>();
}

// u(a, i): component i of the element's vertex a
template <bool APART, typename T, typename U>
__device__ __forceinline__ void element_apply3(const U &u, const T W[27], const GradScale<T> &s, T y[8][3]) {
    T S0[9], S1[9], S2[9];
    pair3<APART, T, 0, 1, true, true, true, true>(u, W, S0, S1, s, y);
    pair3<APART, T, 0, 2, false, true, false, true>(u, W, S0, S2, s, y);
    normal3<APART, T, 0>(u, S0, s, y);
    pair3<APART, T, 1, 2, false, false, true, false>(u, W, S1, S2, s, y);
    normal3<APART, T, 1>(u, S1, s, y);
    normal3<APART, T, 2>(u, S2, s, y);
}

// ---------------------------------------- 2D ----------------------------------------------
// vertex a = bx + 2 by; direction k, orthogonal bit b
__host__ __device__ constexpr int node2(int k, int bk, int b) { return k == 0 ? bk + 2 * b : b + 2 * bk; }

template <typename T, int I, int K>
__device__ __forceinline__ void grad2(const T u[4][2], T sk, T gp[3]) {
    const T d0 = (T)0.5 * sk * (u[node2(K, 1, 0)][I] - u[node2(K, 0, 0)][I]);
    const T d1 = (T)0.5 * sk * (u[node2(K, 1, 1)][I] - u[node2(K, 0, 1)][I]);
    gp[0] = d0;
    gp[1] = (T)0.5 * (d0 + d1);
    gp[2] = d1;
}

template <typename T, int I, int K>
__device__ __forceinline__ void scatter2(const T R[3], T sk, T y[4][2]) {
    const T o0 = R[0] + (T)0.5 * R[1], o1 = R[2] + (T)0.5 * R[1];
    const T v0 = (T)0.5 * sk * o0, v1 = (T)0.5 * sk * o1;
    y[node2(K, 1, 0)][I] += v0;
    y[node2(K, 0, 0)][I] -= v0;
    y[node2(K, 1, 1)][I] += v1;
    y[node2(K, 0, 1)][I] -= v1;
}

template <typename T>
__device__ __forceinline__ void element_apply2(const T u[4][2], const T W[9], const T s[3], T y[4][2]) {
    // diagonal terms: R_ii[q_perp] = 2 gp_ii * sum over q_i of W
    {
        T gp[3], R[3];
        grad2<T, 0, 0>(u, s[0], gp);
#pragma unroll
        for (int q = 0; q < 3; q++) R[q] = (T)2 * gp[q] * (W[0 + 3 * q] + W[1 + 3 * q] + W[2 + 3 * q]);
        scatter2<T, 0, 0>(R, s[0], y);
        grad2<T, 1, 1>(u, s[1], gp);
#pragma unroll
        for (int q = 0; q < 3; q++) R[q] = (T)2 * gp[q] * (W[q] + W[q + 3] + W[q + 6]);
        scatter2<T, 1, 1>(R, s[1], y);
    }
    // shear pair (0,1): tau = W (du0/dx1 + du1/dx0); R_01 sums over q1 (indexed q0), R_10 over q0
    {
        T g01[3], g10[3], R01[3] = {0, 0, 0}, R10[3] = {0, 0, 0};
        grad2<T, 0, 1>(u, s[1], g01);  // indexed by q0
        grad2<T, 1, 0>(u, s[0], g10);  // indexed by q1
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const int q0 = q % 3, q1 = q / 3;
            const T t = W[q] * (g01[q0] + g10[q1]);
            R01[q0] += t;
            R10[q1] += t;
        }
        scatter2<T, 0, 1>(R01, s[1], y);
        scatter2<T, 1, 0>(R10, s[0], y);
    }
}

// ------------------------------------------------------------------------------------------
// Phase 1: one workgroup per tile.  The tile's nodal velocities are staged in LDS, each thread
// applies its element, and the element results are reduced into the tile's node block in LDS.
// Nodes that belong to this tile only are written to y directly; nodes on a face shared with a
// neighbouring tile go to the tile's slot of a workspace.  Phase 2: one thread per shared dof sums
// the 2, 4 or 8 slots that hold it.  No atomics touch global memory and the summation order is
// fixed, so K u is bitwise reproducible.
// ------------------------------------------------------------------------------------------

// does node coordinate gc lie on a face between two tiles along an axis of tile size T (tn tiles)?
__device__ __forceinline__ bool on_tile_face(int gc, int T, int tn) {
    return gc > 0 && gc % T == 0 && gc / T < tn;
}

// What an apply writes for dof i whose product (K u)_i is v (v = 0 on Dirichlet dofs):
//   EPI_Y       y_i = v
//   EPI_RES     y_i = b_i - v, 0 on Dirichlet dofs             (multigrid residual on the free dofs)
//   EPI_CHEBY   r = b_i - v; d_i = c1 d_i + c2 invd_i r; x_i += d_i with x the input u: one Jacobi-
//               Chebyshev smoothing step in place.  In place is safe: a node interior to a tile is
//               staged only by that tile, before its update, and tile-face nodes are updated in
//               phase 2, after every tile has staged them.
//   EPI_CHEBY0  the same with c1 = 0 (the previous d is not read)
//   EPI_PCHEBY0 the multigrid prolongation x += P xc of the coarse-grid correction xc, then the
//               EPI_CHEBY0 step on the corrected x, in one pass: the staged velocities are x + P xc,
//               interpolated from the tile's coarse node block held in LDS (halo kernels: from memory; 2D: halo only).
//   EPI_RES0    the first Jacobi-Chebyshev step from a zero guess, x = c2 invd b, then the residual
//               r = b - K x (0 on Dirichlet dofs), in one pass: the staged velocities are c2 invd b (u is not
//               read); y = r, d = x (the previous d is neither read nor written).
//   EPI_CHEBY1  the first two Jacobi-Chebyshev steps from a zero guess: the staged velocities are x1 = c0 invd b (u is
//               not read), then d = c1 x1 + c2 invd (b - K x1), y = x1 + d.  Halo kernels only.
enum {
    EPI_Y = UST_PASS_Y,
    EPI_RES = UST_PASS_RES,
    EPI_CHEBY = UST_PASS_CHEBY,
    EPI_CHEBY0 = UST_PASS_CHEBY0,
    EPI_PCHEBY0 = UST_PASS_PCHEBY0,
    EPI_RES0 = UST_PASS_RES0,
    EPI_CHEBY1 = UST_PASS_CHEBY1,
    EPI_P = -1  // halo kernels: u is z, staged is the CG direction z + beta p, which goes to next; y as EPI_Y
};
template <typename T>
struct Epi {
    T *y;  // EPI_Y / EPI_RES / EPI_RES0: output; EPI_CHEBY*: x after the step
    const T *b;
    const T *invd;
    T *d;  // EPI_CHEBY*: the Chebyshev direction; EPI_RES0: x after the first step
    T c1, c2;
    const T *xc;  // EPI_PCHEBY0: coarse-grid correction (nodes of the grid with half the elements per axis)
    const T *xs;  // EPI_CHEBY*: x before the step, the input u (y itself when the step runs in place)
    T c0 = (T)0;            // EPI_CHEBY1
    bool d_last = false;    // EPI_CHEBY: no later step reads the direction, leave d as it is
    double *dot = nullptr;  // halo kernels: per workgroup u . y (EPI_Y) or b . x after the step (EPI_CHEBY*), or none
};

__host__ __device__ constexpr bool cheby_mode(int m) { return m == EPI_CHEBY || m == EPI_CHEBY0 || m == EPI_PCHEBY0; }

// (P xc) at fine node (i, j, k): per axis the coarse node i/2 (even i) or the mean of (i-1)/2 and (i+1)/2
// (odd i), trilinear over the axes -- the weights of k_prolong_add.  Branch-free: always 8 terms, the
// second node of an even axis carries weight 0.  cval(I, J, K) returns a coarse value.
template <typename T, typename F>
__device__ __forceinline__ T prolong_value(int i, int j, int k, F cval) {
    const int I0 = i >> 1, J0 = j >> 1, K0 = k >> 1;
    const int I1 = I0 + (i & 1), J1 = J0 + (j & 1), K1 = K0 + (k & 1);
    const T wx = (i & 1) ? (T)0.5 : (T)1, wy = (j & 1) ? (T)0.5 : (T)1, wz = (k & 1) ? (T)0.5 : (T)1;
    const T ox = (i & 1) ? (T)0.5 : (T)0, oy = (j & 1) ? (T)0.5 : (T)0, oz = (k & 1) ? (T)0.5 : (T)0;
    const T a0 = wx * cval(I0, J0, K0) + ox * cval(I1, J0, K0);
    const T a1 = wx * cval(I0, J1, K0) + ox * cval(I1, J1, K0);
    const T a2 = wx * cval(I0, J0, K1) + ox * cval(I1, J0, K1);
    const T a3 = wx * cval(I0, J1, K1) + ox * cval(I1, J1, K1);
    return wz * (wy * a0 + oy * a1) + oz * (wy * a2 + oy * a3);
}

// the same in 2D
template <typename T, typename F>
__device__ __forceinline__ T prolong_value2(int i, int j, F cval) {
    const int I0 = i >> 1, J0 = j >> 1, I1 = I0 + (i & 1), J1 = J0 + (j & 1);
    const T wx = (i & 1) ? (T)0.5 : (T)1, ox = (i & 1) ? (T)0.5 : (T)0;
    const T wy = (j & 1) ? (T)0.5 : (T)1, oy = (j & 1) ? (T)0.5 : (T)0;
    return wy * (wx * cval(I0, J0) + ox * cval(I1, J0)) + oy * (wx * cval(I0, J1) + ox * cval(I1, J1));
}

// the velocity a pass stages for dof i: u, or for EPI_RES0 the first Chebyshev step from zero, c2 invd b
template <int MODE, typename T>
__device__ __forceinline__ T stage_load(const Epi<T> &ep, const T *u, unsigned i) {
    if (MODE == EPI_RES0) return ep.c2 * ep.invd[i] * ep.b[i];
    if (MODE == EPI_CHEBY1) return ep.c0 * ep.invd[i] * ep.b[i];
    return u[i];
}

// operands the epilogue reads, loaded ahead of the stores so that a thread's loads overlap
template <typename T>
struct EpiOps {
    unsigned char m;
    T b, invd, d, x;
};

template <int MODE, typename T>
__device__ __forceinline__ EpiOps<T> epilogue_load(const Epi<T> &ep, const unsigned char *mask, unsigned i) {
    EpiOps<T> o;
    o.m = mask[i];
    o.b = o.invd = o.d = o.x = (T)0;
    if (MODE != EPI_Y && MODE != EPI_P) o.b = ep.b[i];
    if (MODE == EPI_RES0 || MODE == EPI_CHEBY1) o.invd = ep.invd[i];
    if (cheby_mode(MODE)) {
        o.invd = ep.invd[i];
        o.x = ep.xs[i];
    }
    if (MODE == EPI_CHEBY) o.d = ep.d[i];
    return o;
}

// v: the product (K u)_i before masking; returns what goes to y
template <int MODE, typename T>
__device__ __forceinline__ T epilogue_store(const Epi<T> &ep, const EpiOps<T> &o, unsigned i, T v) {
    v = o.m ? (T)0 : v;
    T out;
    if (MODE == EPI_Y || MODE == EPI_P) {
        out = v;
    } else if (MODE == EPI_RES || MODE == EPI_RES0) {
        out = o.m ? (T)0 : o.b - v;
        if (MODE == EPI_RES0) ep.d[i] = ep.c2 * o.invd * o.b;  // as staged (kv_cheby_first's rounding)
    } else {
        const T x = MODE == EPI_CHEBY1 ? ep.c0 * o.invd * o.b : o.x;
        const T d = MODE == EPI_CHEBY1 ? x : o.d;
        const T dn = (MODE == EPI_CHEBY || MODE == EPI_CHEBY1 ? ep.c1 * d : (T)0) + ep.c2 * o.invd * (o.b - v);
        if (ep.d && !ep.d_last) ep.d[i] = dn;  // a first step may come without a d, for the same reason
        out = x + dn;
    }
    ep.y[i] = out;
    return out;
}

// ------------------------------------------------------------------------------------------
// 3D column kernel.  Node plane of a 16x16 column: 17x17 nodes, 867 dofs, NR = 4 per thread.
// ------------------------------------------------------------------------------------------
constexpr int CPX = UST_TX3 + 1, CPY = UST_TY3 + 1, CNP = CPX * CPY, CNPD = CNP * 3;
constexpr int CNR = (CNPD + UST_TILE - 1) / UST_TILE;
// The element-result buffer holds a layer's results with a border of zero elements (18x18 slots per row), so that every
// node sums its four elements per layer at fixed offsets, without a test for the column's edge (row strides of 326 to 342
// measured alike).  With the quotients 2/h taken out of the kernel and the coarse planes of the prolongation interpolated
// once (staged below), a layer took 990 instead of 1400 instructions per thread in the FP32 product and 1200 instead of
// 3150 in the prolongation pass (with an element action of 456 operations; now 606).  128x128x64 passes then, with the
// gather: FP32 product 42.8 -> 38 us, residual with the first step 47.9 -> 44.5, prolongation pass 62.0 -> 54.8, FP64 product
// 73.3 -> 67.3.
constexpr int EBX = UST_TX3 + 2, EBY = UST_TY3 + 2, EBS = 326;
static_assert(EBX * EBY <= EBS && 24 * EBS * 4 % 16 == 0, "18x18 slots per row, cleared by 16-byte stores");

// The column passes' shapes: workgroups per CU the register budget must allow (minb), when the next layer's node plane and
// weights are loaded (pf -- 1: at the start of the layer, held in registers across the element apply; 2: right after the
// element apply, so that they are live only across the reduction and the staging; 0: when they are used), and the
// workgroups the launch aims at, as many as the GPU then holds.  Measured at 128x128x64 (96^3), with the gather, in us:
//   FP32 product      minb 4, pf 0, 1024: 42.0 (39.0)   2, 2, 512: 44.9 (39.1)   3, 2, 768: 44.0 (38.7)
//   FP32 Chebyshev    minb 2, pf 2, 1024: 50.9 (45.2)   4, 0, 1024: 50.7 (46.0; 64^3 21.6 for 20.3)   3, 2, 768: 54.3 (47.3)
//                     (128 registers: four per CU fit)
//   FP32 prolongation minb 3, pf 0, 768: 57.0 (49.6)    2, 2, 512: 59.3 (52.6)   3, 2, 768: 60.8 (53.6)
//                     (four per CU exceed the LDS; with fewer than 768 workgroups of two layers the loads held in
//                     registers are worth more than the third: 64^3 20.5 against 21.9 with an action of 456 operations)
//   FP64 product      minb 2, pf 2, 512: 71.6 (58.0)    2, 0, 512: 85.5 (65.9)   2, 1, 512: 143 (119; spills)
struct ColShape {
    int minb, pf, target;
};
__host__ __device__ constexpr ColShape col_shape(int tsize, int mode, bool many = false) {
    return tsize == 8                                ? ColShape{2, 2, UST_COL_WG_TARGET}
           : mode == EPI_PCHEBY0 && many             ? ColShape{3, 0, UST_COL_WG_TARGET_P}
           : mode == EPI_PCHEBY0                     ? ColShape{2, 2, UST_COL_WG_TARGET}
           : mode == EPI_CHEBY || mode == EPI_CHEBY0 ? ColShape{2, 2, UST_COL_WG_TARGET_F32_YR}
                                                     : ColShape{4, 0, UST_COL_WG_TARGET_F32_YR};
}
// whether the FP32 prolongation pass has workgroups for three per CU
static inline bool col_many(const ust_grid *gr, int tsize, int mode) {
    if (tsize != 4 || mode != EPI_PCHEBY0 || gr->dim != 3) return false;
    const long long cx = (gr->nel[0] + UST_TX3 - 1) / UST_TX3, cy = (gr->nel[1] + UST_TY3 - 1) / UST_TY3;
    return cx * cy * gr->nel[2] >= 2 * UST_COL_WG_TARGET_P;
}
template <typename T, typename WT, int MODE, bool MANY = false>
__global__ __launch_bounds__(256, col_shape(sizeof(T), MODE, MANY).minb) void k_applyK3_col(
    GridDev g, TileDiv td, GradScale<T> gs, const WT *__restrict__ W, const unsigned char *__restrict__ mask, const T *u,
    Epi<T> ep, T *__restrict__ work) {
    __shared__ T su[2][CNPD];     // staged node planes k and k+1 (free dofs; Dirichlet dofs read 0)
    __shared__ __attribute__((aligned(16))) T eb[24 * EBS];  // the layer's results: eb[(a*3 + i)*EBS + slot]
    // EPI_PCHEBY0: a ring of two coarse node planes under the column (9x9 coarse nodes; the column's origin is
    // even, so fine node 2I lies on coarse node I)
    constexpr int CCX = UST_TX3 / 2 + 1, CCY = UST_TY3 / 2 + 1, NCP = CCX * CCY * 3;
    static_assert(NCP <= UST_TILE, "one coarse value per thread");
    __shared__ T sc[MODE == EPI_PCHEBY0 ? 2 * NCP : 1];
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int3 at = tile_at(tile, td);
    const int txy = at.x + g.tnx * at.y, x0 = at.x * UST_TX3, y0 = at.y * UST_TY3;
    const int z0 = at.z * g.tz, z1 = min(z0 + g.tz, g.nz);
    const int tid = threadIdx.x, lx = tid % UST_TX3, ly = tid / UST_TX3;
    const bool active = x0 + lx < g.nx && y0 + ly < g.ny;
    const int es = lx + 1 + EBX * (ly + 1);  // the thread's slot in the element-result buffer
    const unsigned pstride = (unsigned)g.nnx * (unsigned)g.nny * 3u;  // dofs of one global node plane
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1, cnz = g.nz / 2 + 1;  // EPI_PCHEBY0: the coarse grid
    // the plane dofs this thread stages and finishes: t = tid + 256 r -> node n = t / 3 (i = n % 17, j = n / 17),
    // component c = t % 3; pofs = the in-plane part of the global dof index, -1 outside the plane or the grid
    // rofs: the dof's place in the element-result buffer (its upper right element, component c), cofs: in a coarse plane
    int pofs[CNR], rofs[CNR], cofs[MODE == EPI_PCHEBY0 ? CNR : 1];
    bool ring[CNR];
#pragma unroll
    for (int r = 0; r < CNR; r++) {
        const int t = tid + UST_TILE * r, n = t / 3, c = t % 3;
        const int gx = x0 + n % CPX, gy = y0 + n / CPX;
        const bool ok = t < CNPD && gx < g.nnx && gy < g.nny;
        pofs[r] = ok ? (gx + g.nnx * gy) * 3 + c : -1;
        ring[r] = on_tile_face(gx, UST_TX3, g.tnx) || on_tile_face(gy, UST_TY3, g.tny);
        rofs[r] = t < CNPD ? c * EBS + n % CPX + 1 + EBX * (n / CPX + 1) : EBX + 1;
        if (MODE == EPI_PCHEBY0) cofs[r] = t < CNPD ? ((n % CPX / 2) + CCX * (n / CPX / 2)) * 3 + c : 0;
    }
    for (int i = tid; i < (int)(24 * EBS * sizeof(T) / 16); i += UST_TILE) ((float4 *)eb)[i] = float4{0, 0, 0, 0};
    // global loads of plane gz (issued ahead of their use)
    auto load_raw = [&](int gz, T *x, unsigned char *m) {
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            const unsigned dof = pofs[r] >= 0 ? (unsigned)pofs[r] + (unsigned)gz * pstride : 0u;
            m[r] = pofs[r] >= 0 ? mask[dof] : (unsigned char)1;
            x[r] = stage_load<MODE, T>(ep, u, dof);
        }
    };
    // coarse plane c under the column: thread t < NCP loads one value (0 outside the coarse grid)
    auto coarse_load = [&](int c) -> T {
        const int n = tid / 3, cc = tid % 3;
        const int I = x0 / 2 + n % CCX, J = y0 / 2 + n / CCX;
        const bool ok = tid < NCP && I < cnx && J < cny && c < cnz;
        const T v = ep.xc[ok ? ((unsigned)I + (unsigned)cnx * ((unsigned)J + (unsigned)cny * c)) * 3u + cc : 0u];
        return ok ? v : (T)0;
    };
    // staged value: u on free dofs, plus P xc for EPI_PCHEBY0.  The bilinear values of the coarse planes below (pa) and
    // above (pb) the node plane stay in registers: a coarse plane is read from the ring once, by the odd plane under it.
    T pa[MODE == EPI_PCHEBY0 ? CNR : 1], pb[MODE == EPI_PCHEBY0 ? CNR : 1];
    auto coarse_plane = [&](int K, T *v) {
        const T *p = sc + (K & 1) * NCP;
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            const int n = (tid + UST_TILE * r) / 3, i = n % CPX, j = n / CPX;
            const int dx = (i & 1) * 3, dy = (j & 1) * CCX * 3, o = cofs[r];
            const T wx = (i & 1) ? (T)0.5 : (T)1, ox = (i & 1) ? (T)0.5 : (T)0;
            const T wy = (j & 1) ? (T)0.5 : (T)1, oy = (j & 1) ? (T)0.5 : (T)0;
            v[r] = wy * (wx * p[o] + ox * p[o + dx]) + oy * (wx * p[o + dy] + ox * p[o + dx + dy]);
        }
    };
    auto staged = [&](int gz, const T *x, const unsigned char *m, T *v) {
        if (MODE == EPI_PCHEBY0) {
            if (gz & 1) coarse_plane((gz >> 1) + 1, pb);
#pragma unroll
            for (int r = 0; r < CNR; r++) {
                if (!(gz & 1) && gz != z0) pa[r] = pb[r];
                const T pc = (gz & 1) ? (T)0.5 * pa[r] + (T)0.5 * pb[r] : pa[r];
                v[r] = m[r] ? (T)0 : x[r] + pc;
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < CNR; r++) v[r] = m[r] ? (T)0 : x[r];
    };
    // finish plane dof r of global plane gz with value v: the epilogue for a node of this workgroup only, the
    // workspace slot (local plane lp) for a node it shares
    T *slot = work + (size_t)tile * CNP * (g.tz + 1) * 3;
    auto finish = [&](int gz, int lp, bool zshared, const T *planeval, const EpiOps<T> *ops, const T *v) {
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            if (pofs[r] < 0) continue;
            const int t = tid + UST_TILE * r;
            if (ring[r] || zshared) {
                slot[(size_t)lp * CNPD + t] = v[r];
            } else {
                EpiOps<T> o = ops[r];
                if (MODE == EPI_PCHEBY0 && !o.m) o.x = planeval[t];  // x + P xc, as staged
                epilogue_store<MODE, T>(ep, o, (unsigned)pofs[r] + (unsigned)gz * pstride, v[r]);
            }
        }
    };
    auto load_ops = [&](int gz, bool zshared, EpiOps<T> *ops) {
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            const bool own = pofs[r] >= 0 && !ring[r] && !zshared;
            ops[r] = epilogue_load<MODE, T>(ep, mask, own ? (unsigned)pofs[r] + (unsigned)gz * pstride : 0u);
        }
    };
    const size_t wbase = ((size_t)txy * g.nz) * 27 * UST_TILE + tid;
    auto load_w = [&](int k, WT *w) {
#pragma unroll
        for (int q = 0; q < 27; q++) w[q] = W[wbase + ((size_t)k * 27 + q) * UST_TILE];
    };
    // when the next layer's node plane and weights are loaded (col_shape): wpre at the start of this layer,
    // wlate after its element apply; held: in registers (xr, mr, wr) until the next layer uses them
    constexpr int pf = col_shape(sizeof(T), MODE, MANY).pf;
    constexpr bool wpre = pf == 1, wlate = pf == 2, held = pf != 0;
    // ---- prologue: the coarse ring (planes z0/2 and z0/2 + 1), plane z0, and the loads for layer z0 ----
    if (MODE == EPI_PCHEBY0) {
        const int c0 = z0 >> 1;
        const T v0 = coarse_load(c0), v1 = coarse_load(c0 + 1);
        if (tid < NCP) {
            sc[(c0 & 1) * NCP + tid] = v0;
            sc[((c0 + 1) & 1) * NCP + tid] = v1;
        }
        __syncthreads();
        coarse_plane(c0, pa);
    }
    T xr[CNR], carry[CNR];
    unsigned char mr[CNR];
    {
        T v[CNR];
        load_raw(z0, xr, mr);
        staged(z0, xr, mr, v);
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            const int t = tid + UST_TILE * r;
            if (t < CNPD) su[0][t] = v[r];
            carry[r] = (T)0;  // plane z0 receives nothing from below within this chunk
        }
    }
    if (held) load_raw(z0 + 1, xr, mr);
    WT wr[27];
    if (held) load_w(z0, wr);
    // EPI_PCHEBY0: staging an even plane p writes coarse plane p/2 + 1 into the ring (the odd plane p + 1 needs
    // it); its value is loaded one layer ahead
    T cv = (T)0;
    if (MODE == EPI_PCHEBY0 && wpre && ((z0 + 1) & 1) == 0) cv = coarse_load(((z0 + 1) >> 1) + 1);
    // two layers per turn where the next layer's operands are held in registers (FP32 product, loads when used: 38.5 us
    // against 37.9)
#pragma unroll(held ? 2 : 1)
    for (int k = z0; k < z1; k++) {
        const int cur = (k - z0) & 1, nxt = cur ^ 1;
        const bool zsh = k == z0 && z0 > 0;  // the chunk's first plane is shared with the chunk below
        // this layer's operands, loaded during the previous one
        T x1[CNR];
        unsigned char m1[CNR];
        if (held) {
#pragma unroll
            for (int r = 0; r < CNR; r++) {
                x1[r] = xr[r];
                m1[r] = mr[r];
            }
        } else {
            load_raw(k + 1, x1, m1);
        }
        T wq[27];
        if (held) {
#pragma unroll
            for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(wr, q);
        }
        const T cvk = (MODE == EPI_PCHEBY0 && !wpre && ((k + 1) & 1) == 0) ? coarse_load(((k + 1) >> 1) + 1) : cv;
        // the next layer's loads
        if (wpre && k + 2 <= z1) load_raw(k + 2, xr, mr);
        if (wpre && k + 1 < z1) load_w(k + 1, wr);
        if (MODE == EPI_PCHEBY0 && wpre && ((k + 2) & 1) == 0 && k + 1 < z1) cv = coarse_load(((k + 2) >> 1) + 1);
        EpiOps<T> ops[CNR];
        if (wpre) load_ops(k, zsh, ops);
        __syncthreads();  // the previous layer is done with su[nxt], eb and the coarse ring slot written below
        {
            T v[CNR];
            staged(k + 1, x1, m1, v);
#pragma unroll
            for (int r = 0; r < CNR; r++) {
                const int t = tid + UST_TILE * r;
                if (t < CNPD) su[nxt][t] = v[r];
            }
            if (MODE == EPI_PCHEBY0 && ((k + 1) & 1) == 0 && tid < NCP)
                sc[((((k + 1) >> 1) + 1) & 1) * NCP + tid] = cvk;
        }
        __syncthreads();
        {
            if (!held) {
#pragma unroll
                for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(W, wbase + ((size_t)k * 27 + q) * UST_TILE);
            }
            T ye[8][3];
            const T *sb = &su[cur][(lx + CPX * ly) * 3], *st = &su[nxt][(lx + CPX * ly) * 3];
            auto ue = [&](int a, int i) -> T {
                return (a >> 2 ? st : sb)[((a & 1) + CPX * ((a >> 1) & 1)) * 3 + i];
            };
            element_apply3<true, T>(ue, wq, gs, ye);
#pragma unroll
            for (int a = 0; a < 8; a++)
#pragma unroll
                for (int i = 0; i < 3; i++) eb[(a * 3 + i) * EBS + es] = active ? ye[a][i] : (T)0;
        }
        if (wlate && k + 2 <= z1) load_raw(k + 2, xr, mr);
        if (wlate && k + 1 < z1) load_w(k + 1, wr);
        if (!wpre) load_ops(k, zsh, ops);
        __syncthreads();
        // plane k: the carried contributions of layer k-1 plus those of layer k below the plane; the
        // contributions of layer k above plane k+1 become the new carry.  Fixed order, in pairs along x, then y.
        T v[CNR];
#pragma unroll
        for (int r = 0; r < CNR; r++) {
            T lo[4], hi[4];
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const T *e = eb + rofs[r] - (a & 1) - EBX * (a >> 1);
                lo[a] = e[a * 3 * EBS];
                hi[a] = e[(a + 4) * 3 * EBS];
            }
            v[r] = carry[r] + ((lo[3] + lo[2]) + (lo[1] + lo[0]));
            carry[r] = (hi[3] + hi[2]) + (hi[1] + hi[0]);
        }
        finish(k, k - z0, zsh, su[cur], ops, v);
    }
    // the chunk's last plane: shared with the chunk above unless it is the top of the grid
    {
        const bool zsh = z1 < g.nz;
        EpiOps<T> ops[CNR];
        load_ops(z1, zsh, ops);
        finish(z1, z1 - z0, zsh, su[(z1 - z0) & 1], ops, carry);
    }
}

// ------------------------------------------------------------------------------------------
// 3D tile kernel for grids too small for the column kernel to fill the GPU (the coarse multigrid levels):
// one 256-thread workgroup per 16x4x4 tile, one z layer of 64 elements per wavefront, the node block staged
// and reduced in LDS (FP64 accumulation, two wave-parity phases fix the summation order), tile-face nodes
// through the workspace.
// ------------------------------------------------------------------------------------------
template <typename T, typename WT, int MODE>
__global__ __launch_bounds__(256, 2) void k_applyK3_tiled(GridDev g, TileDiv td, GradScale<T> gs,
                                                       const WT *__restrict__ W,
                                                       const unsigned char *__restrict__ mask, const T *u,
                                                       Epi<T> ep, T *__restrict__ work) {
    constexpr int TX = UST_TTX3, TY = UST_TTY3, TZ = UST_TTZ3;
    constexpr int NX = TX + 1, NY = TY + 1, NZ = TZ + 1, NN = NX * NY * NZ;
    __shared__ T su[NN * 3];
    __shared__ double sy[NN * 3];  // FP64 accumulation in LDS for both precisions (ds_add_f64)
    // EPI_PCHEBY0: the coarse nodes under the tile (tile origins are even, so fine node 2I lies on coarse I)
    constexpr int CX = TX / 2 + 1, CY = TY / 2 + 1, CZ = TZ / 2 + 1, NC = CX * CY * CZ * 3;
    static_assert(NC <= UST_TILE, "one coarse value per thread");
    __shared__ T sc[MODE == EPI_PCHEBY0 ? NC : 1];
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int3 at = tile_at(tile, td);
    const int tx0 = at.x * TX, ty0 = at.y * TY, tz0 = at.z * TZ;
    T cv = (T)0;
    if (MODE == EPI_PCHEBY0) {
        const int t = threadIdx.x, c = t % 3, n = t / 3;
        const int I = tx0 / 2 + n % CX, J = ty0 / 2 + (n / CX) % CY, K = tz0 / 2 + n / (CX * CY);
        const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1, cnz = g.nz / 2 + 1;
        const bool ok = t < NC && I < cnx && J < cny && K < cnz;
        cv = ep.xc[ok ? ((unsigned)I + (unsigned)cnx * ((unsigned)J + (unsigned)cny * K)) * 3u + c : 0u];
        cv = ok ? cv : (T)0;
    }
    // Loads are issued without branches, staged velocities first, then the element weights (which do not
    // depend on them), so the LDS stores below wait only for the staging loads and the weights arrive
    // while the tile is being staged.  Out-of-tile slots read dof 0 and are discarded; partial tiles are
    // padded in W, so every load is in bounds.
    constexpr int NST = (NN * 3 + UST_TILE - 1) / UST_TILE;
    T stv[NST];
    bool stok[NST];
    unsigned char stm[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        const int c = t % 3, n = t / 3;
        const int gx = tx0 + n % NX, gy = ty0 + (n / NX) % NY, gz = tz0 + n / (NX * NY);
        stok[r] = t < NN * 3 && gx < g.nnx && gy < g.nny && gz < g.nnz;
        const unsigned dof = stok[r] ? ((unsigned)gx + (unsigned)g.nnx * ((unsigned)gy + (unsigned)g.nny * gz)) * 3u + c : 0u;
        stm[r] = mask[dof];
        stv[r] = stage_load<MODE, T>(ep, u, dof);
    }
    // FP32: the weights are loaded here, ahead of the barrier; FP64 loads them after it, which keeps the
    // register count within two waves per SIMD
    constexpr bool early = sizeof(T) == 4;
    T wq[27];
    if (early) {
#pragma unroll
        for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(W, ((size_t)tile * 27 + q) * UST_TILE + threadIdx.x);
    }
    if (MODE == EPI_PCHEBY0) {
        if (threadIdx.x < NC) sc[threadIdx.x] = cv;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < NST; r++) {
            const int t = threadIdx.x + UST_TILE * r;
            const int c = t % 3, n = t / 3;
            const int ix = n % NX, iy = (n / NX) % NY, iz = n / (NX * NY);
            if (stok[r] && !stm[r])
                stv[r] += prolong_value<T>(ix, iy, iz, [&](int I, int J, int K) {
                    return sc[(I + CX * (J + CY * K)) * 3 + c];
                });
        }
    }
#pragma unroll
    for (int r = 0; r < NST; r++) stv[r] = (stok[r] && !stm[r]) ? stv[r] : (T)0;
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        if (t < NN * 3) {
            su[t] = stv[r];
            sy[t] = 0.0;
        }
    }
    __syncthreads();
    const int lx = threadIdx.x % TX, ly = (threadIdx.x / TX) % TY, lz = threadIdx.x / (TX * TY);
    const bool active = tx0 + lx < g.nx && ty0 + ly < g.ny && tz0 + lz < g.nz;
    T ye[8][3];
    if (active) {
        if (!early) {
#pragma unroll
            for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(W, ((size_t)tile * 27 + q) * UST_TILE + threadIdx.x);
        }
        const T *sb = &su[(lx + NX * (ly + NY * lz)) * 3];
        element_apply3<false, T>([&](int a, int i) -> T {
            return sb[((a & 1) + NX * (((a >> 1) & 1) + NY * (a >> 2))) * 3 + i];
        }, wq, gs, ye);
    }
    // Wave w holds the element layer lz = w, whose nodes are layers w and w+1: even waves never share a
    // node, nor do odd waves, and within one LDS add the 64 lanes hit 64 distinct nodes.  Adding in two
    // wave-parity phases therefore fixes the order in which every node receives its contributions.
    for (int phase = 0; phase < 2; phase++) {
        if (active && (lz & 1) == phase) {
#pragma unroll
            for (int a = 0; a < 8; a++) {
                const int ln = (lx + (a & 1)) + NX * ((ly + ((a >> 1) & 1)) + NY * (lz + (a >> 2)));
#pragma unroll
                for (int i = 0; i < 3; i++) atomicAdd(&sy[ln * 3 + i], (double)ye[a][i]);
            }
        }
        __syncthreads();
    }
    // writeout: every load of the thread (mask, epilogue operands) first, then the stores.  Dof indices are
    // 32-bit (the host rejects larger grids), which keeps the per-thread index registers down.
    T *slot = work + (size_t)tile * NN * 3;
    int kind[NST];  // 0 none, 1 tile-face node (workspace slot), 2 node of this tile only (written here)
    unsigned wdof[NST];
    EpiOps<T> ops[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        const int c = t % 3, n = t / 3;
        const int gx = tx0 + n % NX, gy = ty0 + (n / NX) % NY, gz = tz0 + n / (NX * NY);
        const bool in = t < NN * 3 && gx < g.nnx && gy < g.nny && gz < g.nnz;
        const bool face = on_tile_face(gx, TX, g.tnx) || on_tile_face(gy, TY, g.tny) || on_tile_face(gz, TZ, g.tnz);
        kind[r] = in ? (face ? 1 : 2) : 0;
        wdof[r] = kind[r] == 2 ? ((unsigned)gx + (unsigned)g.nnx * ((unsigned)gy + (unsigned)g.nny * gz)) * 3u + c : 0u;
        ops[r] = epilogue_load<MODE, T>(ep, mask, wdof[r]);
    }
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        if (MODE == EPI_PCHEBY0 && kind[r] == 2 && !ops[r].m) ops[r].x = su[t];  // x + P xc, as staged
        if (kind[r] == 1) slot[t] = (T)sy[t];
        else if (kind[r] == 2) epilogue_store<MODE, T>(ep, ops[r], wdof[r], (T)sy[t]);
    }
}

// ------------------------------------------------------------------------------------------
// Halo kernels: a 256-thread workgroup owns a block of NODES and computes every element touching them -- in 3D an 8x4x4
// block and its 9x5x5 elements (a one-element halo on the low side of each axis), in 2D 15x15 nodes and 16x16 elements,
// one element per thread -- so every owned node's sum is complete inside the workgroup: one launch, no workspace and no
// gather.  The halo elements are computed by two workgroups, which costs less on the latency-bound grids than the gather
// it replaces.  Neighbouring workgroups stage the nodes a workgroup writes, so the Chebyshev modes must run out of place
// (ep.xs != ep.y).  Each node sums its element contributions in a fixed order, in FP64: deterministic.  The operands of the
// epilogue are loaded with the node block, so that only one trip to memory is exposed, and a pass can leave per-workgroup
// partial sums of the dot product that follows it in the Krylov iteration.
// What bounds them is the serial chain of one wavefront: launch, one trip to memory, 1300-1800 instructions, a store.  With
// every pass of such levels on them an inner iteration took 14 launches in 2D at 64x64 where tiles + gather, separate first
// steps, prolongation and dots took 24; solves: 2D 64x64 FP64 129.6 -> 74.7 ms, 3D 24x16x16 FP64 661 -> 455 ms.
// Staging whole nodes (index arithmetic once per node, none of the loads behind a branch) instead of single dofs:
// 466.8 -> 455 ms of the latter, the 64x64x32 solve with FP32 PCG 388 -> 379 ms.
// ------------------------------------------------------------------------------------------
constexpr int HOX = 8, HOY = 4, HOZ = 4;                    // owned nodes per axis
constexpr int HEX = HOX + 1, HEY = HOY + 1, HEZ = HOZ + 1;  // element slots per axis
constexpr int HNX = HOX + 2, HNY = HOY + 2, HNZ = HOZ + 2;  // staged nodes per axis
constexpr int HNE = HEX * HEY * HEZ, HNN = HNX * HNY * HNZ;  // 225 element slots, 360 staged nodes
static_assert(HNE <= UST_TILE && HOX * HOY * HOZ * 2 == UST_TILE, "one element, at most two owned dofs per thread");
constexpr int H2O = 15, H2N = H2O + 2, H2D = H2O * H2O * 2;  // 2D: owned nodes and staged nodes per axis, owned dofs

// EPI_P: the previous direction p, the new one next, and the CG's control block and partial sums (ust_cg.h)
template <typename T>
struct CgDir {
    const T *p;
    T *next;
    double *c;
    const double *part;
    int nrz, nrr;
};
// the direction's beta, or false once the CG has stopped; called by every thread of the workgroup, whose first one writes
// the control block
template <typename T>
__device__ __forceinline__ bool cg_direction(const CgDir<T> &cg, bool *first, T *beta) {
    const CgSums s = cg_sums(cg.part + CG_RZ, cg.nrz, cg.part + CG_RR, cg.nrr, cg.c);
    double thr = 0.0;
    const double state = cg_state(s, s.b, &thr);
    if (blockIdx.x == 0 && threadIdx.x == 0 && s.c[1] == 0.0) {
        cg.c[1] = state;
        cg.c[2] = s.c[4];
        cg.c[3] = s.a;
        cg.c[6] = thr;
    }
    *first = s.c[4] == 0.0;
    *beta = (T)(s.a / s.c[5]);
    return state == 0.0;
}

// 3D grids up to this many elements may take the halo kernel: the 128x128x64 solve takes 0.403-0.407 s with the halo passes
// on its 32x32x16 and 16x16x8 levels (0.431-0.434 without) and 0.415-0.417 s with them on the 64x64x32 level as well.
#ifndef UST_HALO_MAX_NEL
#define UST_HALO_MAX_NEL 65536
#endif
// A CU works through its halo workgroups one after the other (FP64 product: 5.2 us with up to 256 of them, 7.3 up to 512,
// 10.5 beyond), through a tile and the gather in about 9.3, two tiles in 10.9.  So beyond 512 workgroups grids of at most one
// tile per CU take tiles.  FP64 product, halo / tiles: 36^3 7.4 / 9.1 us, 48x36x36 10.4 / 9.3, 64x32x32 10.6 / 9.5, 40^3 (300
// tiles) 10.6 / 10.8, 65x33x30 (360) 10.5 / 11.0; FP32 prolongation pass 36^3 10.4 / 10.7, 64x32x32 14.5 / 11.0.  Solves of
// 64x32x32 in FP64 837 / 814 ms, with FP32 PCG 300 / 281; 128x64x64 539 / 526.
// 2D grids take it whatever their size: one element in seven is computed again, where the gather was half of a pass.  FP64
// product 256^2 3.9 / 6.8 us, 512x256 4.2 / 7.3, 1000^2 17.1 / 25.8, 1500^2 34.2 / 53; FP32 1000^2 12.4 / 19.8.
constexpr int HALO_FULL = 512, HALO_CUS = 256;

__host__ __device__ inline int halo_tiles(const GridDev &g) {
    if (g.dim == 2) return ((g.nnx + H2O - 1) / H2O) * ((g.nny + H2O - 1) / H2O);
    return ((g.nnx + HOX - 1) / HOX) * ((g.nny + HOY - 1) / HOY) * ((g.nnz + HOZ - 1) / HOZ);
}
static inline bool halo_grid(const GridDev &g) {
    if (g.dim == 2) return true;
    return !g.col && g.nel <= UST_HALO_MAX_NEL && (halo_tiles(g) <= HALO_FULL || g.ntiles > HALO_CUS);
}

// whether a pass writes a vector that it stages, at nodes that other workgroups own: u, or for the steps from zero b and
// invd, and the coarse correction.  (Those an owned node alone reads may be written over.)
template <int MODE, typename T>
static inline bool writes_staged(const Epi<T> &ep, const T *u) {
    const bool zero = MODE == EPI_RES0 || MODE == EPI_CHEBY1;
    const T *staged[3] = {zero ? ep.b : u, zero ? ep.invd : nullptr, MODE == EPI_PCHEBY0 ? ep.xc : nullptr};
    for (const T *v : staged)
        if (v && (ep.y == v || ep.d == v)) return true;
    return false;
}

// the workgroup's sum of v into out[block]
__device__ __forceinline__ void block_dot(double v, double *out) {
    __shared__ double sh[4];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// the contributions v(a) of the elements that have a node as vertex a, in pairs along x, then y, then z: fewer roundings than
// one after the other, and no more operations
template <typename V>
__device__ __forceinline__ double vertex_sum3(V v) {
    const double lo = (v(3) + v(2)) + (v(1) + v(0)), hi = (v(7) + v(6)) + (v(5) + v(4));
    return hi + lo;
}

template <typename T, typename WT, int MODE>
__global__ __launch_bounds__(256) void k_applyK3_halo(GridDev g, TileDiv td, GradScale<T> gs,
                                                      const WT *__restrict__ W,
                                                      const unsigned char *__restrict__ mask, const T *u, Epi<T> ep,
                                                      CgDir<T> cg) {
    __shared__ T su[HNN * 3];   // staged node block, origin (nx0 - 1, ny0 - 1, nz0 - 1)
    __shared__ T eb[24 * HNE];  // element results: eb[(a*3 + i) * HNE + slot] (HNE odd: rows shift banks)
    const int tile = xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int3 at = tile_at(tile, td);
    const int nx0 = at.x * HOX, ny0 = at.y * HOY, nz0 = at.z * HOZ;
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1;  // EPI_PCHEBY0: the coarse grid
    // staging: two nodes per thread, the three components together; nodes outside the grid stage 0 (their loads go to the
    // nearest node of the grid, so that none of them waits for a branch)
    constexpr int NST = (HNN + UST_TILE - 1) / UST_TILE;
    T stv[NST][3];
    T stp[MODE == EPI_P ? NST : 1][3];
    unsigned char stm[NST][3];
    bool stok[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        const int gx = nx0 - 1 + n % HNX, gy = ny0 - 1 + (n / HNX) % HNY, gz = nz0 - 1 + n / (HNX * HNY);
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1), kz = min(max(gz, 0), g.nnz - 1);
        stok[r] = gx == kx && gy == ky && gz == kz;
        const unsigned dof = ((unsigned)kx + (unsigned)g.nnx * ((unsigned)ky + (unsigned)g.nny * kz)) * 3u;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            stm[r][c] = mask[dof + c];
            stv[r][c] = stage_load<MODE, T>(ep, u, dof + c);
            if (MODE == EPI_P) stp[r][c] = cg.p[dof + c];
        }
        if (MODE == EPI_PCHEBY0) {  // x + P xc on the free dofs, the coarse values read from global memory
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const T pc = prolong_value<T>(kx, ky, kz, [&](int I, int J, int K) {
                    return ep.xc[((unsigned)I + (unsigned)cnx * ((unsigned)J + (unsigned)cny * K)) * 3u + c];
                });
                stv[r][c] += stm[r][c] ? (T)0 : pc;
            }
        }
    }
    // the thread's element slot and its weights, loaded while the block is staged
    const int lx = tid % HEX, ly = (tid / HEX) % HEY, lz = tid / (HEX * HEY);
    const int ex = nx0 - 1 + lx, ey = ny0 - 1 + ly, ez = nz0 - 1 + lz;
    const bool valid = tid < HNE && ex >= 0 && ey >= 0 && ez >= 0 && ex < g.nx && ey < g.ny && ez < g.nz;
    const size_t w0 = valid ? widx_at(g, ex, ey, ez, 0) : 0;
    T wq[27];
#pragma unroll
    for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(W, w0 + (size_t)q * UST_TILE);
    // the owned dofs: node tid % 128 of the block, component tid / 128 and, for the first 128 threads, component 2
    const int on = tid % (HOX * HOY * HOZ), ox = on % HOX, oy = (on / HOX) % HOY, oz = on / (HOX * HOY);
    const bool inside = nx0 + ox < g.nnx && ny0 + oy < g.nny && nz0 + oz < g.nnz;
    const unsigned odof =
        inside ? ((unsigned)(nx0 + ox) + (unsigned)g.nnx * ((unsigned)(ny0 + oy) + (unsigned)g.nny * (nz0 + oz))) * 3u
               : 0u;
    EpiOps<T> ops[2];
#pragma unroll
    for (int r = 0; r < 2; r++) ops[r] = epilogue_load<MODE, T>(ep, mask, odof + (r ? 2 : tid / (HOX * HOY * HOZ)));
    if (MODE == EPI_P) {
        bool first;
        T beta;
        if (!cg_direction(cg, &first, &beta)) return;
#pragma unroll
        for (int r = 0; r < NST; r++) {
            const int n = tid + UST_TILE * r;
            const int ax = n % HNX, ay = (n / HNX) % HNY, az = n / (HNX * HNY);
            const bool mine = stok[r] && ax >= 1 && ax <= HOX && ay >= 1 && ay <= HOY && az >= 1 && az <= HOZ && n < HNN;
            const unsigned row = (unsigned)(ny0 - 1 + ay) + (unsigned)g.nny * (nz0 - 1 + az);
            const unsigned dof = ((unsigned)(nx0 - 1 + ax) + (unsigned)g.nnx * row) * 3u;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                stv[r][c] = first ? stv[r][c] : stv[r][c] + beta * stp[r][c];
                if (mine) cg.next[dof + c] = stv[r][c];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        if (n < HNN)
#pragma unroll
            for (int c = 0; c < 3; c++) su[n * 3 + c] = (stok[r] && !stm[r][c]) ? stv[r][c] : (T)0;
    }
    __syncthreads();
    if (tid < HNE) {
        T ye[8][3];
        const T *sb = &su[(lx + HNX * (ly + HNY * lz)) * 3];
        element_apply3<false, T>([&](int a, int i) -> T {
            return sb[((a & 1) + HNX * (((a >> 1) & 1) + HNY * (a >> 2))) * 3 + i];
        }, wq, gs, ye);
#pragma unroll
        for (int a = 0; a < 8; a++)
#pragma unroll
            for (int i = 0; i < 3; i++) eb[(a * 3 + i) * HNE + tid] = valid ? ye[a][i] : (T)0;
    }
    __syncthreads();
    // each owned dof sums its 8 elements in a fixed order, then the epilogue
    double dot = 0.0;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        if (!inside || (r && tid >= HOX * HOY * HOZ)) continue;
        const int c = r ? 2 : tid / (HOX * HOY * HOZ);
        const T us = su[((ox + 1) + HNX * ((oy + 1) + HNY * (oz + 1))) * 3 + c];
        const double v = vertex_sum3([&](int a) {  // element slot (ox + 1 - dx, ...) has this node as vertex (dx, dy, dz)
            return (double)eb[(a * 3 + c) * HNE + (ox + 1 - (a & 1)) + HEX * ((oy + 1 - ((a >> 1) & 1)) +
                                                                              HEY * (oz + 1 - (a >> 2)))];
        });
        EpiOps<T> o = ops[r];
        if (MODE == EPI_PCHEBY0 && !o.m) o.x = us;  // x + P xc, as staged
        const T out = epilogue_store<MODE, T>(ep, o, odof + c, (T)v);
        dot += (double)out * (double)(MODE == EPI_Y || MODE == EPI_P ? us : o.b);
    }
    if (ep.dot) block_dot(dot, ep.dot);
}

template <typename T, typename WT, int MODE>
__global__ __launch_bounds__(256) void k_applyK2_halo(GridDev g, TileDiv td, const WT *__restrict__ W,
                                                      const unsigned char *__restrict__ mask, const T *u, Epi<T> ep,
                                                      CgDir<T> cg) {
    __shared__ T su[H2N * H2N * 2];          // staged node block, origin (nx0 - 1, ny0 - 1)
    __shared__ T eb[8 * (UST_TILE + 1)];     // element results: eb[(a*2 + i) * 257 + slot]
    const int tile = xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int3 at = tile_at(tile, td);
    const int nx0 = at.x * H2O, ny0 = at.y * H2O;
    const int cnx = g.nx / 2 + 1;  // EPI_PCHEBY0: the coarse grid
    constexpr int NSN = H2N * H2N, NST = (NSN + UST_TILE - 1) / UST_TILE;
    T stv[NST][2];
    T stp[MODE == EPI_P ? NST : 1][2];
    unsigned char stm[NST][2];
    bool stok[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        const int gx = nx0 - 1 + n % H2N, gy = ny0 - 1 + n / H2N;
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1);
        stok[r] = gx == kx && gy == ky;
        const unsigned dof = ((unsigned)kx + (unsigned)g.nnx * (unsigned)ky) * 2u;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            stm[r][c] = mask[dof + c];
            stv[r][c] = stage_load<MODE, T>(ep, u, dof + c);
            if (MODE == EPI_P) stp[r][c] = cg.p[dof + c];
        }
        if (MODE == EPI_PCHEBY0) {
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const T pc = prolong_value2<T>(kx, ky, [&](int I, int J) {
                    return ep.xc[((unsigned)I + (unsigned)cnx * (unsigned)J) * 2u + c];
                });
                stv[r][c] += stm[r][c] ? (T)0 : pc;
            }
        }
    }
    const int lx = tid % 16, ly = tid / 16, ex = nx0 - 1 + lx, ey = ny0 - 1 + ly;
    const bool valid = ex >= 0 && ey >= 0 && ex < g.nx && ey < g.ny;
    const size_t w0 = valid ? widx_at(g, ex, ey, 0, 0) : 0;
    T wq[9];
#pragma unroll
    for (int q = 0; q < 9; q++) wq[q] = wload<T, WT>(W, w0 + (size_t)q * UST_TILE);
    EpiOps<T> ops[2];
    unsigned dofs[2];
    bool own[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int d = tid + UST_TILE * r, n = d / 2;
        const int gx = nx0 + n % H2O, gy = ny0 + n / H2O;
        own[r] = d < H2D && gx < g.nnx && gy < g.nny;
        dofs[r] = own[r] ? ((unsigned)gx + (unsigned)g.nnx * (unsigned)gy) * 2u + d % 2 : 0u;
        ops[r] = epilogue_load<MODE, T>(ep, mask, dofs[r]);
    }
    if (MODE == EPI_P) {
        bool first;
        T beta;
        if (!cg_direction(cg, &first, &beta)) return;
#pragma unroll
        for (int r = 0; r < NST; r++) {
            const int n = tid + UST_TILE * r;
            const int ax = n % H2N, ay = n / H2N;
            const bool mine = stok[r] && ax >= 1 && ax <= H2O && ay >= 1 && ay <= H2O && n < NSN;
            const unsigned dof = ((unsigned)(nx0 - 1 + ax) + (unsigned)g.nnx * (unsigned)(ny0 - 1 + ay)) * 2u;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                stv[r][c] = first ? stv[r][c] : stv[r][c] + beta * stp[r][c];
                if (mine) cg.next[dof + c] = stv[r][c];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        if (n < NSN)
#pragma unroll
            for (int c = 0; c < 2; c++) su[n * 2 + c] = (stok[r] && !stm[r][c]) ? stv[r][c] : (T)0;
    }
    __syncthreads();
    {
        T ue[4][2], ye[4][2];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int ln = (lx + (a & 1)) + H2N * (ly + (a >> 1));
            ue[a][0] = su[ln * 2];
            ue[a][1] = su[ln * 2 + 1];
            ye[a][0] = ye[a][1] = (T)0;
        }
        const T s[3] = {(T)g.sx, (T)g.sy, (T)1};
        element_apply2<T>(ue, wq, s, ye);
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int i = 0; i < 2; i++) eb[(a * 2 + i) * (UST_TILE + 1) + tid] = valid ? ye[a][i] : (T)0;
    }
    __syncthreads();
    double dot = 0.0;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        if (!own[r]) continue;
        const int d = tid + UST_TILE * r, n = d / 2, c = d % 2, ox = n % H2O, oy = n / H2O;
        const T us = su[((ox + 1) + H2N * (oy + 1)) * 2 + c];
        double v = 0.0;
#pragma unroll
        for (int dy = 1; dy >= 0; dy--)
#pragma unroll
            for (int dx = 1; dx >= 0; dx--)  // element slot (ox + 1 - dx, oy + 1 - dy) has this node as vertex (dx, dy)
                v += (double)eb[((dx + 2 * dy) * 2 + c) * (UST_TILE + 1) + (ox + 1 - dx) + 16 * (oy + 1 - dy)];
        EpiOps<T> o = ops[r];
        if (MODE == EPI_PCHEBY0 && !o.m) o.x = us;  // x + P xc, as staged
        const T out = epilogue_store<MODE, T>(ep, o, dofs[r], (T)v);
        dot += (double)out * (double)(MODE == EPI_Y || MODE == EPI_P ? us : o.b);
    }
    if (ep.dot) block_dot(dot, ep.dot);
}

// ------------------------------------------------------------------------------------------
// Fused level passes: the pre-smoothing of a level with its residual and restriction, and in 2D both post-smoothing steps,
// in one launch.  A workgroup owns a block of coarse nodes (of nodes, for the post-smoothing) and computes what they depend
// on, one or two rings of elements around the block: more arithmetic, but on the grids that take the halo kernels a launch
// and its trip to memory cost more.  With the direction formed by the product's pass, an inner iteration takes 7 launches
// for 14 at 2D 64x64 and 11 for 14 at 3D 24x16x16.  Solves: 2D 64x64 FP64 74.2 -> 54.4 ms, 256x256 117 -> 70, 512x256
// 181 -> 113; 3D 24x16x16 FP64 453 -> 431, 64x64x32 with FP32 PCG (two such levels) 368 -> 363.5.
// Every value is computed by the formulas and in the order of the separate passes.
// ------------------------------------------------------------------------------------------
// 2D, three kinds: residual of u; of the first step from zero; of the first two steps from zero.  6x6 coarse nodes, that is
// 13x13 residual nodes, 14x14 elements, 15x15 nodes of x, and one more ring for the kind whose x takes a product.
constexpr int F2C = 6, F2R = 2 * F2C + 1, F2X = F2R + 2, F2S = F2X + 2, F2E = 16;
static_assert(F2S == F2E + 1 && F2E * F2E == UST_TILE, "one element per thread");
enum { PRE_U = 0, PRE_FIRST = 1, PRE_TWO = 2 };

// the element of this thread's slot applied to the staged block su into eb; slots outside the grid leave zeros
template <typename T>
__device__ __forceinline__ void block_apply2(const T *su, int lx, int ly, bool valid, const T *wq, const T *s, T *eb) {
    T ue[4][2], ye[4][2];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const int ln = (lx + (a & 1)) + F2S * (ly + (a >> 1));
        ue[a][0] = su[ln * 2];
        ue[a][1] = su[ln * 2 + 1];
        ye[a][0] = ye[a][1] = (T)0;
    }
    element_apply2<T>(ue, wq, s, ye);
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int i = 0; i < 2; i++) eb[(a * 2 + i) * (UST_TILE + 1) + lx + F2E * ly] = valid ? ye[a][i] : (T)0;
}
// (K x) at node (i, j) of the 15x15 ring, component c
template <typename T>
__device__ __forceinline__ T block_sum2(const T *eb, int i, int j, int c) {
    double v = 0.0;
#pragma unroll
    for (int dy = 1; dy >= 0; dy--)
#pragma unroll
        for (int dx = 1; dx >= 0; dx--)
            v += (double)eb[((dx + 2 * dy) * 2 + c) * (UST_TILE + 1) + (i + 1 - dx) + F2E * (j + 1 - dy)];
    return (T)v;
}

template <typename T, typename WT, int KIND>
__global__ __launch_bounds__(256) void k_pre2(GridDev g, TileDiv td, const WT *__restrict__ W,
                                              const unsigned char *__restrict__ mask,
                                              const unsigned char *__restrict__ maskc, const T *__restrict__ u,
                                              const T *__restrict__ b, const T *__restrict__ invd, T *__restrict__ y,
                                              T *__restrict__ d, T *__restrict__ bc, T c0, T c1, T c2) {
    __shared__ T su[F2S * F2S * 2];
    __shared__ T eb[8 * (UST_TILE + 1)];
    __shared__ T sr[F2R * F2R * 2];
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1;
    const int tile = xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int3 at = tile_at(tile, td);
    const int I0 = at.x * F2C, J0 = at.y * F2C;
    const int ox = 2 * I0 - 3, oy = 2 * J0 - 3;  // origin of the staged block
    const auto dof_of = [&](int gx, int gy, bool *in) -> unsigned {
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1);
        *in = kx == gx && ky == gy;
        return ((unsigned)kx + (unsigned)g.nnx * (unsigned)ky) * 2u;
    };
    // the first x at the staged nodes
    constexpr int NST = (F2S * F2S + UST_TILE - 1) / UST_TILE;
    T sv[NST][2];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = min(tid + UST_TILE * r, F2S * F2S - 1);
        bool in;
        const unsigned k = dof_of(ox + n % F2S, oy + n / F2S, &in);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const bool m = mask[k + c] != 0;
            const T x = KIND == PRE_U ? u[k + c] : (KIND == PRE_FIRST ? c2 : c0) * invd[k + c] * b[k + c];
            sv[r][c] = in && !m ? x : (T)0;
        }
    }
    // the thread's element and its weights, and its node of the 15x15 ring
    const int lx = tid % F2E, ly = tid / F2E, ex = ox + lx, ey = oy + ly;
    const bool valid = ex >= 0 && ey >= 0 && ex < g.nx && ey < g.ny;
    const size_t w0 = valid ? widx_at(g, ex, ey, 0, 0) : 0;
    T wq[9];
#pragma unroll
    for (int q = 0; q < 9; q++) wq[q] = wload<T, WT>(W, w0 + (size_t)q * UST_TILE);
    const bool node = tid < F2X * F2X;
    const int i = min(tid, F2X * F2X - 1) % F2X, j = min(tid, F2X * F2X - 1) / F2X;
    bool in;
    const unsigned k = dof_of(ox + 1 + i, oy + 1 + j, &in);
    const bool own = node && in && i >= 2 && j >= 2 && i < 2 + 2 * F2C && j < 2 + 2 * F2C;
    bool m[2];
    T bv[2], iv[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        m[c] = mask[k + c] != 0;
        bv[c] = b[k + c];
        iv[c] = KIND == PRE_U ? (T)0 : invd[k + c];
    }
    const int cn = tid / 2, cc = tid % 2, I = I0 + cn % F2C, J = J0 + cn / F2C;
    const bool coarse = tid < F2C * F2C * 2 && I < cnx && J < cny;
    const unsigned ck = coarse ? ((unsigned)I + (unsigned)cnx * (unsigned)J) * 2u + cc : 0u;
    const bool mc = maskc[ck] != 0;
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        if (n < F2S * F2S) {
            su[n * 2] = sv[r][0];
            su[n * 2 + 1] = sv[r][1];
        }
    }
    const T s[3] = {(T)g.sx, (T)g.sy, (T)1};
    __syncthreads();
    block_apply2(su, lx, ly, valid, wq, s, eb);
    __syncthreads();
    if (KIND == PRE_TWO) {
        if (node) {
            T x2[2];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const T v = m[c] ? (T)0 : block_sum2(eb, i, j, c);
                const T x = c0 * iv[c] * bv[c];
                const T dn = c1 * x + c2 * iv[c] * (bv[c] - v);
                x2[c] = x + dn;
                if (own) {
                    y[k + c] = x2[c];
                    if (d) d[k + c] = dn;
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++) su[((i + 1) + F2S * (j + 1)) * 2 + c] = in && !m[c] ? x2[c] : (T)0;
        }
        __syncthreads();
        block_apply2(su, lx, ly, valid, wq, s, eb);  // the outer ring of slots is not used any more
        __syncthreads();
    }
    if (KIND == PRE_FIRST && own) {
#pragma unroll
        for (int c = 0; c < 2; c++) d[k + c] = c2 * iv[c] * bv[c];
    }
    if (node && i >= 1 && j >= 1 && i <= F2R && j <= F2R) {
#pragma unroll
        for (int c = 0; c < 2; c++)
            sr[((i - 1) + F2R * (j - 1)) * 2 + c] = in && !m[c] ? bv[c] - block_sum2(eb, i, j, c) : (T)0;
    }
    __syncthreads();
    if (!coarse) return;
    const int ci = 2 * (I - I0) + 1, cj = 2 * (J - J0) + 1;
    T acc = (T)0;
#pragma unroll
    for (int dy = -1; dy <= 1; dy++)
#pragma unroll
        for (int dx = -1; dx <= 1; dx++)
            acc += (T)((dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0)) * sr[((ci + dx) + F2R * (cj + dy)) * 2 + cc];
    bc[ck] = mc ? (T)0 : acc;
}

// 2D, both post-smoothing steps: 13x13 nodes
template <typename T, typename WT>
__global__ __launch_bounds__(256) void k_post2(GridDev g, TileDiv td, const WT *__restrict__ W,
                                              const unsigned char *__restrict__ mask,
                                               const T *__restrict__ u, const T *__restrict__ xc, const T *__restrict__ b,
                                               const T *__restrict__ invd, T *__restrict__ y, T c0, T c1, T c2,
                                               double *__restrict__ dots) {
    __shared__ T su[F2S * F2S * 2];
    __shared__ T eb[8 * (UST_TILE + 1)];
    const int cnx = g.nx / 2 + 1;
    const int tile = xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int3 at = tile_at(tile, td);
    const int ox = at.x * F2R - 2, oy = at.y * F2R - 2;  // origin of the staged block
    const auto dof_of = [&](int gx, int gy, bool *in) -> unsigned {
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1);
        *in = kx == gx && ky == gy;
        return ((unsigned)kx + (unsigned)g.nnx * (unsigned)ky) * 2u;
    };
    constexpr int NST = (F2S * F2S + UST_TILE - 1) / UST_TILE;
    T sv[NST][2];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = min(tid + UST_TILE * r, F2S * F2S - 1);
        const int gx = ox + n % F2S, gy = oy + n / F2S;
        bool in;
        const unsigned k = dof_of(gx, gy, &in);
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const bool m = mask[k + c] != 0;
            const T pc = prolong_value2<T>(kx, ky, [&](int I, int J) {
                return xc[((unsigned)I + (unsigned)cnx * (unsigned)J) * 2u + c];
            });
            const T x = u[k + c] + pc;
            sv[r][c] = in && !m ? x : (T)0;
        }
    }
    const int lx = tid % F2E, ly = tid / F2E, ex = ox + lx, ey = oy + ly;
    const bool valid = ex >= 0 && ey >= 0 && ex < g.nx && ey < g.ny;
    const size_t w0 = valid ? widx_at(g, ex, ey, 0, 0) : 0;
    T wq[9];
#pragma unroll
    for (int q = 0; q < 9; q++) wq[q] = wload<T, WT>(W, w0 + (size_t)q * UST_TILE);
    const bool node = tid < F2X * F2X;
    const int i = min(tid, F2X * F2X - 1) % F2X, j = min(tid, F2X * F2X - 1) / F2X;
    bool in;
    const unsigned k = dof_of(ox + 1 + i, oy + 1 + j, &in);
    bool m[2];
    T bv[2], iv[2], uv[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        m[c] = mask[k + c] != 0;
        bv[c] = b[k + c];
        iv[c] = invd[k + c];
        uv[c] = u[k + c];
    }
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int n = tid + UST_TILE * r;
        if (n < F2S * F2S) {
            su[n * 2] = sv[r][0];
            su[n * 2 + 1] = sv[r][1];
        }
    }
    const T s[3] = {(T)g.sx, (T)g.sy, (T)1};
    __syncthreads();
    block_apply2(su, lx, ly, valid, wq, s, eb);
    __syncthreads();
    T x1[2], d1[2];
    if (node) {
        const int sn = ((i + 1) + F2S * (j + 1)) * 2;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const T v = m[c] ? (T)0 : block_sum2(eb, i, j, c);
            const T x = m[c] ? uv[c] : su[sn + c];
            d1[c] = c0 * iv[c] * (bv[c] - v);
            x1[c] = x + d1[c];
        }
#pragma unroll
        for (int c = 0; c < 2; c++) su[sn + c] = in && !m[c] ? x1[c] : (T)0;
    }
    __syncthreads();
    block_apply2(su, lx, ly, valid, wq, s, eb);
    __syncthreads();
    double dot = 0.0;
    if (node && in && i >= 1 && j >= 1 && i <= F2R && j <= F2R) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const T v = m[c] ? (T)0 : block_sum2(eb, i, j, c);
            const T dn = c1 * d1[c] + c2 * iv[c] * (bv[c] - v);
            const T out = x1[c] + dn;
            y[k + c] = out;
            dot += (double)out * (double)bv[c];
        }
    }
    if (dots) block_dot(dot, dots);
}

// 3D, residual of u or of the first step from zero: 3x2x2 coarse nodes, that is 7x5x5 residual nodes, 8x6x6 elements (one
// per thread of 320), 9x7x7 staged nodes.
constexpr int F3X = 3, F3Y = 2, F3Z = 2;                                      // coarse nodes
constexpr int F3RX = 2 * F3X + 1, F3RY = 2 * F3Y + 1, F3RZ = 2 * F3Z + 1;     // residual nodes
constexpr int F3EX = F3RX + 1, F3EY = F3RY + 1, F3EZ = F3RZ + 1;              // elements
constexpr int F3SX = F3EX + 1, F3SY = F3EY + 1, F3SZ = F3EZ + 1;              // staged nodes
constexpr int F3E = F3EX * F3EY * F3EZ, F3R = F3RX * F3RY * F3RZ, F3S = F3SX * F3SY * F3SZ, F3T = 320;
static_assert(F3E <= F3T && F3R * 3 <= 2 * F3T && F3S <= 2 * F3T, "288 elements, 525 residual dofs, 441 nodes");

template <typename T, typename WT, int KIND>
__global__ __launch_bounds__(F3T) void k_pre3(GridDev g, TileDiv td, GradScale<T> gs, const WT *__restrict__ W,
                                              const unsigned char *__restrict__ mask,
                                              const unsigned char *__restrict__ maskc, const T *__restrict__ u,
                                              const T *__restrict__ b, const T *__restrict__ invd, T *__restrict__ d,
                                              T *__restrict__ bc, T c2) {
    constexpr int EB = F3E + 1;
    __shared__ T su[F3S * 3];
    __shared__ T eb[24 * EB];
    __shared__ T sr[F3R * 3];
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1, cnz = g.nz / 2 + 1;
    const int tile = xcd_block(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int3 at = tile_at(tile, td);
    const int I0 = at.x * F3X, J0 = at.y * F3Y, K0 = at.z * F3Z;
    const int ox = 2 * I0 - 2, oy = 2 * J0 - 2, oz = 2 * K0 - 2;  // origin of the staged block and of the elements
    const auto dof_of = [&](int gx, int gy, int gz, bool *in) -> unsigned {
        const int kx = min(max(gx, 0), g.nnx - 1), ky = min(max(gy, 0), g.nny - 1), kz = min(max(gz, 0), g.nnz - 1);
        *in = kx == gx && ky == gy && kz == gz;
        return ((unsigned)kx + (unsigned)g.nnx * ((unsigned)ky + (unsigned)g.nny * kz)) * 3u;
    };
    T sv[2][3];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int n = min(tid + F3T * r, F3S - 1);
        bool in;
        const unsigned k = dof_of(ox + n % F3SX, oy + (n / F3SX) % F3SY, oz + n / (F3SX * F3SY), &in);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const bool m = mask[k + c] != 0;
            const T x = KIND == PRE_U ? u[k + c] : c2 * invd[k + c] * b[k + c];
            sv[r][c] = in && !m ? x : (T)0;
        }
    }
    const int et = min(tid, F3E - 1), lx = et % F3EX, ly = (et / F3EX) % F3EY, lz = et / (F3EX * F3EY);
    const int ex = ox + lx, ey = oy + ly, ez = oz + lz;
    const bool valid = ex >= 0 && ey >= 0 && ez >= 0 && ex < g.nx && ey < g.ny && ez < g.nz;
    const size_t w0 = valid ? widx_at(g, ex, ey, ez, 0) : 0;
    T wq[27];
#pragma unroll
    for (int q = 0; q < 27; q++) wq[q] = wload<T, WT>(W, w0 + (size_t)q * UST_TILE);
    // the residual dofs t = tid, tid + 320: component t / 175 of node t % 175
    bool rin[2], rm[2];
    T rb[2], ri[2];
    unsigned rk[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int t = min(tid + F3T * r, F3R * 3 - 1), c = t / F3R, n = t % F3R;
        rk[r] = dof_of(ox + 1 + n % F3RX, oy + 1 + (n / F3RX) % F3RY, oz + 1 + n / (F3RX * F3RY), &rin[r]) + c;
        rm[r] = mask[rk[r]] != 0;
        rb[r] = b[rk[r]];
        ri[r] = KIND == PRE_U ? (T)0 : invd[rk[r]];
    }
    const int cn = tid / 3, cc = tid % 3;
    const int I = I0 + cn % F3X, J = J0 + (cn / F3X) % F3Y, K = K0 + cn / (F3X * F3Y);
    const bool coarse = tid < F3X * F3Y * F3Z * 3 && I < cnx && J < cny && K < cnz;
    const unsigned ck = coarse ? ((unsigned)I + (unsigned)cnx * ((unsigned)J + (unsigned)cny * K)) * 3u + cc : 0u;
    const bool mc = maskc[ck] != 0;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int n = tid + F3T * r;
        if (n < F3S)
#pragma unroll
            for (int c = 0; c < 3; c++) su[n * 3 + c] = sv[r][c];
    }
    __syncthreads();
    if (tid < F3E) {
        T ye[8][3];
        const T *sb = &su[(lx + F3SX * (ly + F3SY * lz)) * 3];
        element_apply3<false, T>([&](int a, int q) -> T {
            return sb[((a & 1) + F3SX * (((a >> 1) & 1) + F3SY * (a >> 2))) * 3 + q];
        }, wq, gs, ye);
#pragma unroll
        for (int a = 0; a < 8; a++)
#pragma unroll
            for (int q = 0; q < 3; q++) eb[(a * 3 + q) * EB + tid] = valid ? ye[a][q] : (T)0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int t = tid + F3T * r;
        if (t >= F3R * 3) continue;
        const int c = t / F3R, n = t % F3R, i = n % F3RX, j = (n / F3RX) % F3RY, k = n / (F3RX * F3RY);
        const double v = vertex_sum3([&](int a) {
            return (double)eb[(a * 3 + c) * EB + (i + 1 - (a & 1)) + F3EX * ((j + 1 - ((a >> 1) & 1)) +
                                                                           F3EY * (k + 1 - (a >> 2)))];
        });
        sr[n * 3 + c] = rin[r] && !rm[r] ? rb[r] - (T)v : (T)0;
        // x = the first step, on the nodes 2 I0 .. 2 I0 + 5 and so on, each of one workgroup
        if (KIND == PRE_FIRST && rin[r] && i >= 1 && j >= 1 && k >= 1) d[rk[r]] = c2 * ri[r] * rb[r];
    }
    __syncthreads();
    if (!coarse) return;
    const int ci = 2 * (I - I0) + 1, cj = 2 * (J - J0) + 1, cq = 2 * (K - K0) + 1;
    T acc = (T)0;
#pragma unroll
    for (int dz = -1; dz <= 1; dz++)
#pragma unroll
        for (int dy = -1; dy <= 1; dy++)
#pragma unroll
            for (int dx = -1; dx <= 1; dx++)
                acc += (T)((dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0) * (dz ? 0.5 : 1.0)) *
                       sr[((ci + dx) + F3RX * ((cj + dy) + F3RY * (cq + dz))) * 3 + cc];
    bc[ck] = mc ? (T)0 : acc;
}

static int fused_groups(const GridDev &g, int mode) {
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1, cnz = g.nz / 2 + 1;
    if (mode == UST_PASS_PCHEBY2) return ((g.nnx + F2R - 1) / F2R) * ((g.nny + F2R - 1) / F2R);
    if (g.dim == 2) return ((cnx + F2C - 1) / F2C) * ((cny + F2C - 1) / F2C);
    return ((cnx + F3X - 1) / F3X) * ((cny + F3Y - 1) / F3Y) * ((cnz + F3Z - 1) / F3Z);
}

template <typename T, typename WT>
static int fused_pass(const GridDev &g, const ust_pass *p, hipStream_t st) {
    const T *u = (const T *)p->u, *b = (const T *)p->b, *invd = (const T *)p->invd;
    T *y = (T *)p->y, *d = (T *)p->d, *bc = (T *)p->bc;
    const WT *W = (const WT *)p->W;
    const T c0 = (T)p->c0, c1 = (T)p->c1, c2 = (T)p->c2;
    const int mode = p->mode;
    if (!W || !p->mask || !b) return UST_EINVAL;
    if (g.nx % 2 || g.ny % 2 || (g.dim == 3 && g.nz % 2)) return UST_EINVAL;
    if (g.dim == 3 && mode != UST_PASS_RESR && mode != UST_PASS_RES0R) return UST_EINVAL;
    if (mode != UST_PASS_RESR && !invd) return UST_EINVAL;
    if (mode != UST_PASS_PCHEBY2 && (!bc || !p->maskc)) return UST_EINVAL;
    if ((mode == UST_PASS_RESR || mode == UST_PASS_PCHEBY2) && !u) return UST_EINVAL;
    if (mode == UST_PASS_RES0R && !d) return UST_EINVAL;
    if (mode == UST_PASS_CHEBY1R && !y) return UST_EINVAL;
    if (mode == UST_PASS_PCHEBY2 && (!y || !p->xc)) return UST_EINVAL;
    // every vector read is read at nodes that other workgroups own, and what is written is written once
    const bool from_u = mode == UST_PASS_RESR || mode == UST_PASS_PCHEBY2, post = mode == UST_PASS_PCHEBY2;
    const void *in[4] = {b, from_u ? u : nullptr, mode == UST_PASS_RESR ? nullptr : invd, post ? p->xc : nullptr};
    const void *out[3] = {post || mode == UST_PASS_CHEBY1R ? y : nullptr,
                          mode == UST_PASS_RES0R || mode == UST_PASS_CHEBY1R ? d : nullptr, post ? nullptr : bc};
    for (int i = 0; i < 3; i++) {
        for (int k = 0; k < 4; k++)
            if (out[i] && out[i] == in[k]) return UST_EINVAL;
        if (out[i] && out[i] == out[(i + 1) % 3]) return UST_EINVAL;
    }
    const dim3 grid(fused_groups(g, mode));
    const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1;
    const TileDiv td = mode == UST_PASS_PCHEBY2 ? tile_div((g.nnx + F2R - 1) / F2R, (g.nny + F2R - 1) / F2R)
                       : g.dim == 2             ? tile_div((cnx + F2C - 1) / F2C, (cny + F2C - 1) / F2C)
                                                : tile_div((cnx + F3X - 1) / F3X, (cny + F3Y - 1) / F3Y);
#define PRE2(KIND) hipLaunchKernelGGL((k_pre2<T, WT, KIND>), grid, dim3(UST_TILE), 0, st, g, td, W, p->mask, p->maskc, u, b, \
                                      invd, y, d, bc, c0, c1, c2)
#define PRE3(KIND) hipLaunchKernelGGL((k_pre3<T, WT, KIND>), grid, dim3(F3T), 0, st, g, td, grad_scale<T>(g), W, p->mask, \
                                      p->maskc, u, b, invd, d, bc, c2)
    if (mode == UST_PASS_PCHEBY2)
        hipLaunchKernelGGL((k_post2<T, WT>), grid, dim3(UST_TILE), 0, st, g, td, W, p->mask, u, (const T *)p->xc, b, invd, y,
                           c0, c1, c2, p->dot);
    else if (g.dim == 3 && mode == UST_PASS_RESR) PRE3(PRE_U);
    else if (g.dim == 3) PRE3(PRE_FIRST);
    else if (mode == UST_PASS_RESR) PRE2(PRE_U);
    else if (mode == UST_PASS_RES0R) PRE2(PRE_FIRST);
    else PRE2(PRE_TWO);
#undef PRE2
#undef PRE3
    UST_LAUNCH_CHECK();
    return UST_OK;
}

template <typename T, typename WT, int MODE>
__global__ __launch_bounds__(256) void k_applyK2_tiled(GridDev g, TileDiv td, const WT *__restrict__ W,
                                                       const unsigned char *__restrict__ mask, const T *u,
                                                       Epi<T> ep, T *__restrict__ work) {
    constexpr int TX = UST_TX2, TY = UST_TY2;
    constexpr int NX = TX + 1, NY = TY + 1, NN = NX * NY;
    __shared__ T su[NN * 2];
    __shared__ double sy[NN * 2];
    const int tile = blockIdx.x;
    const int3 at = tile_at(tile, td);
    const int tx0 = at.x * TX, ty0 = at.y * TY;
    constexpr int NST = (NN * 2 + UST_TILE - 1) / UST_TILE;
    T stv[NST];
    bool stok[NST];
    unsigned char stm[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        const int c = t % 2, n = t / 2;
        const int gx = tx0 + n % NX, gy = ty0 + n / NX;
        stok[r] = t < NN * 2 && gx < g.nnx && gy < g.nny;
        const unsigned dof = stok[r] ? ((unsigned)gx + (unsigned)g.nnx * gy) * 2u + c : 0u;
        stm[r] = mask[dof];
        stv[r] = stage_load<MODE, T>(ep, u, dof);
    }
    T wq[9];
#pragma unroll
    for (int q = 0; q < 9; q++) wq[q] = wload<T, WT>(W, ((size_t)tile * 9 + q) * UST_TILE + threadIdx.x);
#pragma unroll
    for (int r = 0; r < NST; r++) stv[r] = (stok[r] && !stm[r]) ? stv[r] : (T)0;
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        if (t < NN * 2) {
            su[t] = stv[r];
            sy[t] = 0.0;
        }
    }
    __syncthreads();
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const bool active = tx0 + lx < g.nx && ty0 + ly < g.ny;
    T ye[4][2];
    if (active) {
        T ue[4][2];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int ln = (lx + (a & 1)) + NX * (ly + (a >> 1));
            ue[a][0] = su[ln * 2];
            ue[a][1] = su[ln * 2 + 1];
            ye[a][0] = ye[a][1] = (T)0;
        }
        const T s[3] = {(T)g.sx, (T)g.sy, (T)1};
        element_apply2<T>(ue, wq, s, ye);
    }
    // wave w holds element rows 4w..4w+3 (node rows 4w..4w+4): same two-phase ordering as in 3D
    const int wave = threadIdx.x / 64;
    for (int phase = 0; phase < 2; phase++) {
        if (active && (wave & 1) == phase) {
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const int ln = (lx + (a & 1)) + NX * (ly + (a >> 1));
                atomicAdd(&sy[ln * 2], (double)ye[a][0]);
                atomicAdd(&sy[ln * 2 + 1], (double)ye[a][1]);
            }
        }
        __syncthreads();
    }
    T *slot = work + (size_t)tile * NN * 2;
    int kind[NST];
    unsigned wdof[NST];
    EpiOps<T> ops[NST];
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        const int c = t % 2, n = t / 2;
        const int gx = tx0 + n % NX, gy = ty0 + n / NX;
        const bool in = t < NN * 2 && gx < g.nnx && gy < g.nny;
        const bool face = on_tile_face(gx, TX, g.tnx) || on_tile_face(gy, TY, g.tny);
        kind[r] = in ? (face ? 1 : 2) : 0;
        wdof[r] = kind[r] == 2 ? ((unsigned)gx + (unsigned)g.nnx * gy) * 2u + c : 0u;
        ops[r] = epilogue_load<MODE, T>(ep, mask, wdof[r]);
    }
#pragma unroll
    for (int r = 0; r < NST; r++) {
        const int t = threadIdx.x + UST_TILE * r;
        if (kind[r] == 1) slot[t] = (T)sy[t];
        else if (kind[r] == 2) epilogue_store<MODE, T>(ep, ops[r], wdof[r], (T)sy[t]);
    }
}

// Phase 2 visits only the nodes on tile faces, enumerated as three disjoint regular sets so that every
// thread has work: Z = the z-face planes (all x, y), Y = the y-face planes off the z-faces, X = the
// x-face lines off both.  An axis with tn tiles has tn - 1 face coordinates T, 2T, ..., (tn-1)T.
template <int DIM>
static inline unsigned face_node_count(const GridDev &g) {
    const unsigned fx = g.tnx - 1, fy = g.tny - 1, fz = DIM == 3 ? g.tnz - 1 : 0;
    return fz * g.nnx * g.nny + fy * g.nnx * (g.nnz - fz) + fx * (g.nny - fy) * (g.nnz - fz);
}

struct GatherDiv {  // divisors of the face enumeration: nodes per row and column, faces, off-face rows, z tile and z tile - 1
    FastDiv nnx, nny, fx, fy, ny, tz, tz1;
};
static inline GatherDiv gather_div(const GridDev &g) {
    const auto one = [](int v) { return fast_div(v < 1 ? 1u : (unsigned)v); };
    return {one(g.nnx), one(g.nny), one(g.tnx - 1), one(g.tny - 1), one(g.nny - (g.tny - 1)), one(g.tz), one(g.tz - 1)};
}

// k-th coordinate that is not a tile face: 0, 1..T-1, T+1..2T-1, ..., (tn-1)T+1 .. end; blk = (k - 1) / (T - 1)
__device__ __forceinline__ int nonface_coord(int k, int T, int tn, int blk) {
    if (k == 0) return 0;
    blk = min(blk, tn - 1);
    return 1 + blk * T + (k - 1 - blk * (T - 1));
}

// A thread per dof of the faces.  The work is index arithmetic: with the divisors known only at run time as plain integer
// divisions, 540 instructions per thread bound the 128x128x64 passes at 9.7-13.3 us; as products with precomputed
// reciprocals and the tile sizes known at compile time it is a third of that.
template <typename T, int DIM, int MODE, bool COL>
__global__ __launch_bounds__(256) void k_gather_tiles(GridDev g, GatherDiv q, const unsigned char *__restrict__ mask,
                                                      const T *__restrict__ work, Epi<T> ep) {
    constexpr int TX = DIM == 2 ? UST_TX2 : COL ? UST_TX3 : UST_TTX3, TY = DIM == 2 ? UST_TY2 : COL ? UST_TY3 : UST_TTY3;
    const int TZ = DIM == 2 ? 1 : COL ? g.tz : UST_TTZ3;
    constexpr int NX = TX + 1, NY = TY + 1;
    const unsigned NN = NX * NY * (DIM == 3 ? TZ + 1 : 1);
    const int fx = g.tnx - 1, fy = g.tny - 1, fz = DIM == 3 ? g.tnz - 1 : 0;
    const unsigned nZ = (unsigned)fz * g.nnx * g.nny;
    const unsigned nY = (unsigned)fy * g.nnx * (g.nnz - fz);
    const unsigned nX = (unsigned)fx * (g.nny - fy) * (g.nnz - fz);
    const unsigned tt = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = (int)(tt % DIM);
    unsigned t = tt / DIM;
    const auto nonface_z = [&](unsigned k) {
        return nonface_coord((int)k, TZ, g.tnz, k == 0 ? 0 : (int)(COL ? (k - 1) / q.tz1 : (k - 1) / (UST_TTZ3 - 1)));
    };
    int gx, gy, gz;
    if (t < nZ) {
        const unsigned r = t / q.nnx, p = r / q.nny;
        gx = (int)(t - r * g.nnx);
        gy = (int)(r - p * g.nny);
        gz = TZ * (int)(p + 1);
    } else if ((t -= nZ) < nY) {
        const unsigned r = t / q.nnx, p = r / q.fy;
        gx = (int)(t - r * g.nnx);
        gy = TY * (int)(r - p * fy + 1);
        gz = DIM == 3 ? nonface_z(p) : 0;
    } else if ((t -= nY) < nX) {
        const unsigned r = t / q.fx, p = r / q.ny;
        const int j = (int)(r - p * q.ny.d);
        gx = TX * (int)(t - r * fx + 1);
        gy = nonface_coord(j, TY, g.tny, (j - 1) / (TY - 1));
        gz = DIM == 3 ? nonface_z(p) : 0;
    } else {
        return;
    }
    const unsigned n = (unsigned)gx + (unsigned)g.nnx * ((unsigned)gy + (unsigned)g.nny * gz);
    EpiOps<T> ops = epilogue_load<MODE, T>(ep, mask, n * DIM + c);
    // the tiles that hold the node, the upper one first along each axis, and its place in them
    const int tx = min(gx / TX, g.tnx - 1), ty = min(gy / TY, g.tny - 1);
    const int tz = DIM == 2 ? 0 : min((int)(COL ? (unsigned)gz / q.tz : (unsigned)gz / UST_TTZ3), g.tnz - 1);
    const int lx = gx - tx * TX, ly = gy - ty * TY, lz = gz - tz * TZ;
    const bool sx = lx == 0 && tx > 0, sy = ly == 0 && ty > 0, sz = DIM == 3 && lz == 0 && tz > 0;
    const T *slot = work + ((size_t)((unsigned)tx + (unsigned)g.tnx * ((unsigned)ty + (unsigned)g.tny * tz)) * NN +
                            (unsigned)(lx + NX * (ly + NY * lz))) * DIM + c;
    // steps to the lower tile of an axis, at its last node
    const ptrdiff_t dx = ((ptrdiff_t)TX - (ptrdiff_t)NN) * DIM;
    const ptrdiff_t dy = ((ptrdiff_t)NX * TY - (ptrdiff_t)g.tnx * NN) * DIM;
    const ptrdiff_t dz = ((ptrdiff_t)NX * NY * TZ - (ptrdiff_t)g.tnx * g.tny * NN) * DIM;
    T v[8];
#pragma unroll
    for (int a = 0; a < (DIM == 3 ? 8 : 4); a++) {
        const bool have = (!(a & 1) || sx) && (!(a & 2) || sy) && (!(a & 4) || sz);
        v[a] = have ? slot[(a & 1 ? dx : 0) + (a & 2 ? dy : 0) + (a & 4 ? dz : 0)] : (T)0;
    }
    T acc = (T)0;
#pragma unroll
    for (int a = 0; a < (DIM == 3 ? 8 : 4); a++) acc += v[a];
    if (MODE == EPI_PCHEBY0 && !ops.m) {  // 3D only (host-checked): x + P xc on a free component
        const int cnx = g.nx / 2 + 1, cny = g.ny / 2 + 1;
        ops.x += prolong_value<T>(gx, gy, gz, [&](int I, int J, int K) {
            return ep.xc[((unsigned)I + (unsigned)cnx * ((unsigned)J + (unsigned)cny * K)) * 3u + c];
        });
    }
    epilogue_store<MODE, T>(ep, ops, n * DIM + c, acc);
}

template <typename T, int DIM, int MODE, bool COL>
static void gather_tiles(const GridDev &g, const unsigned char *mask, const T *work, const Epi<T> &ep, hipStream_t st) {
    const unsigned nf = face_node_count<DIM>(g);
    if (nf)
        hipLaunchKernelGGL((k_gather_tiles<T, DIM, MODE, COL>), dim3(ust_grid_size((size_t)nf * DIM, 256)), dim3(256), 0,
                           st, g, gather_div(g), mask, work, ep);
}

static inline size_t work_len(const GridDev &g) {
    const size_t nn = g.dim == 3 ? (size_t)(g.tx + 1) * (g.ty + 1) * (g.tz + 1) : (size_t)(g.tx + 1) * (g.ty + 1);
    return (size_t)g.ntiles * nn * g.dim;
}

template <typename T, typename WT, int MODE>
static int apply_halo(const GridDev &g, const WT *W, const unsigned char *mask, const T *u, const Epi<T> &ep,
                      hipStream_t st, const CgDir<T> &cg = {}) {
    if (g.dim == 3)
        hipLaunchKernelGGL((k_applyK3_halo<T, WT, MODE>), dim3(halo_tiles(g)), dim3(UST_TILE), 0, st, g,
                           tile_div((g.nnx + HOX - 1) / HOX, (g.nny + HOY - 1) / HOY), grad_scale<T>(g), W, mask, u, ep, cg);
    else
        hipLaunchKernelGGL((k_applyK2_halo<T, WT, MODE>), dim3(halo_tiles(g)), dim3(UST_TILE), 0, st, g,
                           tile_div((g.nnx + H2O - 1) / H2O, (g.nny + H2O - 1) / H2O), W, mask, u, ep, cg);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

template <typename T, typename WT, int MODE>
static int apply_tiled(const ust_grid *gr, const WT *W, const unsigned char *mask, const T *u, Epi<T> ep, T *work,
                       void *stream) {
    const bool many = col_many(gr, sizeof(T), MODE);
    GridDev g = grid_dev(gr, col_shape(sizeof(T), MODE, many).target);
    const TileDiv td = tile_div(g.tnx, g.tny);
    if (!W || !mask || !u || !ep.y || !work) return UST_EINVAL;
    if (MODE != EPI_Y && !ep.b) return UST_EINVAL;
    if (cheby_mode(MODE) && (!ep.invd || (MODE == EPI_CHEBY && !ep.d) || ep.xs != u)) return UST_EINVAL;
    if (MODE == EPI_RES0 && (!ep.invd || !ep.d)) return UST_EINVAL;
    if (MODE == EPI_PCHEBY0 && (g.dim != 3 || !ep.xc || g.nx % 2 || g.ny % 2 || g.nz % 2)) return UST_EINVAL;
    if ((size_t)g.nnx * g.nny * g.nnz * g.dim >= (1ull << 32)) return UST_EINVAL;  // 32-bit dof indices
    hipStream_t st = ust_stream(stream);
    // small 3D grids and 2D ones: the halo kernel, unless the pass overwrites what its neighbours stage (a Chebyshev step, a
    // product or a residual in place, a first step over its right-hand side), which tiles + gather allow
    if (halo_grid(g) && !writes_staged<MODE>(ep, u)) return apply_halo<T, WT, MODE>(g, W, mask, u, ep, st);
    if (g.dim == 3) {
        const GradScale<T> gs = grad_scale<T>(g);
        if (g.col) {
            if constexpr (sizeof(T) == 4 && MODE == EPI_PCHEBY0)
                if (many)
                    hipLaunchKernelGGL((k_applyK3_col<T, WT, MODE, true>), dim3(g.ntiles), dim3(UST_TILE), 0, st, g, td, gs,
                                       W, mask, u, ep, work);
            if (!many)
                hipLaunchKernelGGL((k_applyK3_col<T, WT, MODE>), dim3(g.ntiles), dim3(UST_TILE), 0, st, g, td, gs, W,
                                   mask, u, ep, work);
            gather_tiles<T, 3, MODE, true>(g, mask, work, ep, st);
        } else {
            hipLaunchKernelGGL((k_applyK3_tiled<T, WT, MODE>), dim3(g.ntiles), dim3(UST_TILE), 0, st, g, td, gs, W, mask,
                               u, ep, work);
            gather_tiles<T, 3, MODE, false>(g, mask, work, ep, st);
        }
    } else {
        hipLaunchKernelGGL((k_applyK2_tiled<T, WT, MODE>), dim3(g.ntiles), dim3(UST_TILE), 0, st, g, td, W, mask, u, ep,
                           work);
        gather_tiles<T, 2, MODE, false>(g, mask, work, ep, st);
    }
    UST_LAUNCH_CHECK();
    return UST_OK;
}

template <typename T, typename WT>
static int apply_plain(const ust_grid *g, const WT *W, const unsigned char *mask, const T *u, T *y, T *work,
                       void *stream) {
    Epi<T> ep = {y, nullptr, nullptr, nullptr, (T)0, (T)0, nullptr, nullptr};
    return apply_tiled<T, WT, EPI_Y>(g, W, mask, u, ep, work, stream);
}

template <typename T, typename WT>
static int apply_residual(const ust_grid *g, const WT *W, const unsigned char *mask, const T *u, const T *b, T *r,
                          T *work, void *stream) {
    Epi<T> ep = {r, b, nullptr, nullptr, (T)0, (T)0, nullptr, nullptr};
    return apply_tiled<T, WT, EPI_RES>(g, W, mask, u, ep, work, stream);
}

// xi: x before the step; x: after it (the same vector when the step runs in place)
template <typename T, typename WT>
static int apply_cheby(const ust_grid *g, const WT *W, const unsigned char *mask, const T *xi, T *x, const T *b,
                       const T *invd, T *d, T c1, T c2, int first, T *work, void *stream) {
    Epi<T> ep = {x, b, invd, d, c1, c2, nullptr, xi};
    return first ? apply_tiled<T, WT, EPI_CHEBY0>(g, W, mask, xi, ep, work, stream)
                 : apply_tiled<T, WT, EPI_CHEBY>(g, W, mask, xi, ep, work, stream);
}

template <typename T, typename WT>
static int apply_cheby_prolong(const ust_grid *g, const WT *W, const unsigned char *mask, const T *xi, T *x,
                               const T *b, const T *invd, T *d, T c2, const T *xc, T *work, void *stream) {
    Epi<T> ep = {x, b, invd, d, (T)0, c2, xc, xi};
    return apply_tiled<T, WT, EPI_PCHEBY0>(g, W, mask, xi, ep, work, stream);
}

template <typename T, typename WT>
static int apply_residual_first(const ust_grid *g, const WT *W, const unsigned char *mask, const T *b, const T *invd,
                                T *x, T *r, T c2, T *work, void *stream) {
    Epi<T> ep = {r, b, invd, x, (T)0, c2, nullptr, nullptr};
    return apply_tiled<T, WT, EPI_RES0>(g, W, mask, b, ep, work, stream);  // u unused: b stands in
}

extern "C" int ust_k_apply_K_residual_first_f32(const ust_grid *g, const float *WK, const unsigned char *mask,
                                                const float *b, const float *invd, float *x, float *r, float c2,
                                                float *work, void *stream) {
    return apply_residual_first<float, float>(g, WK, mask, b, invd, x, r, c2, work, stream);
}

// One halo pass from its description.
template <typename T, typename WT>
static int halo_pass(const GridDev &g, const ust_pass *p, hipStream_t st) {
    const T *u = (const T *)p->u, *b = (const T *)p->b, *invd = (const T *)p->invd, *xc = (const T *)p->xc;
    T *y = (T *)p->y, *d = (T *)p->d;
    const WT *W = (const WT *)p->W;
    if (p->mode >= UST_PASS_RESR && p->mode <= UST_PASS_PCHEBY2) return fused_pass<T, WT>(g, p, st);
    Epi<T> ep = {y, b, invd, d, (T)p->c1, (T)p->c2, xc, u, (T)p->c0, p->d_last != 0, p->dot};
    if (!W || !p->mask || !y) return UST_EINVAL;
    const bool reads_u = p->mode != UST_PASS_RES0 && p->mode != UST_PASS_CHEBY1;
    if (reads_u && !u) return UST_EINVAL;
    if (p->mode != UST_PASS_Y && !b) return UST_EINVAL;
    if (p->mode >= UST_PASS_CHEBY && !invd) return UST_EINVAL;
    if (!reads_u) u = b;  // not read
    if (p->mode <= UST_PASS_RES) ep.d = nullptr;  // not written
    // out of place
#define HALO(MODE) return writes_staged<MODE>(ep, u) ? UST_EINVAL : apply_halo<T, WT, MODE>(g, W, p->mask, u, ep, st)
    switch (p->mode) {
        case UST_PASS_Y: HALO(EPI_Y);
        case UST_PASS_RES: HALO(EPI_RES);
        case UST_PASS_CHEBY:
            if (!d) return UST_EINVAL;
            HALO(EPI_CHEBY);
        case UST_PASS_CHEBY0: HALO(EPI_CHEBY0);
        case UST_PASS_PCHEBY0:
            if (!xc || g.nx % 2 || g.ny % 2 || (g.dim == 3 && g.nz % 2)) return UST_EINVAL;
            HALO(EPI_PCHEBY0);
        case UST_PASS_RES0:
            if (!d) return UST_EINVAL;
            HALO(EPI_RES0);
        case UST_PASS_CHEBY1: HALO(EPI_CHEBY1);
    }
#undef HALO
    return UST_EINVAL;
}

extern "C" int ust_k_apply_single(const ust_grid *gr) {
    const GridDev g = grid_dev(gr);
    return halo_grid(g) ? halo_tiles(g) : 0;
}

extern "C" int ust_k_apply_groups(const ust_grid *gr, int mode) {
    const GridDev g = grid_dev(gr);
    if (!halo_grid(g)) return 0;
    return mode >= UST_PASS_RESR && mode <= UST_PASS_PCHEBY2 ? fused_groups(g, mode) : halo_tiles(g);
}

extern "C" int ust_k_cg_dir_apply(const ust_grid *gr, int type, const void *W, const unsigned char *mask, const void *z,
                                  const void *p, void *next, void *q, double *c, double *part, int nrz, size_t n,
                                  void *stream) {
    if (!gr || !W || !mask || !z || !p || !next || !q || !c || !part || nrz < 1 || nrz > UST_CG_PARTS) return UST_EINVAL;
    if (next == z || next == p || q == z || q == p || q == next) return UST_EINVAL;
    const GridDev g = grid_dev(gr);
    if (!halo_grid(g) || halo_tiles(g) > UST_CG_PARTS) return UST_EINVAL;
    if (n != (size_t)g.nnx * g.nny * g.nnz * g.dim || n >= (1ull << 32)) return UST_EINVAL;
    hipStream_t st = ust_stream(stream);
    const int nrr = ust_k_cg_parts(n);
    if (type == UST_PASS_F64) {
        const CgDir<double> cg = {(const double *)p, (double *)next, c, part, nrz, nrr};
        const Epi<double> ep = {(double *)q, nullptr, nullptr, nullptr, 0.0, 0.0, nullptr, nullptr, 0.0, false, part + CG_PQ};
        return apply_halo<double, double, EPI_P>(g, (const double *)W, mask, (const double *)z, ep, st, cg);
    }
    if (type == UST_PASS_F32) {
        const CgDir<float> cg = {(const float *)p, (float *)next, c, part, nrz, nrr};
        const Epi<float> ep = {(float *)q, nullptr, nullptr, nullptr, 0.0f, 0.0f, nullptr, nullptr, 0.0f, false,
                               part + CG_PQ};
        return apply_halo<float, float, EPI_P>(g, (const float *)W, mask, (const float *)z, ep, st, cg);
    }
    return UST_EINVAL;
}

extern "C" int ust_k_apply_pass(const ust_grid *gr, const ust_pass *p, void *stream) {
    if (!gr || !p) return UST_EINVAL;
    const GridDev g = grid_dev(gr);
    if (!halo_grid(g)) return UST_EINVAL;
    if ((size_t)g.nnx * g.nny * g.nnz * g.dim >= (1ull << 32)) return UST_EINVAL;  // 32-bit dof indices
    hipStream_t st = ust_stream(stream);
    if (p->type == UST_PASS_F64) return halo_pass<double, double>(g, p, st);
    if (p->type == UST_PASS_F32) return halo_pass<float, float>(g, p, st);
    if (p->type == UST_PASS_F32_BF16W) return halo_pass<float, unsigned short>(g, p, st);
    return UST_EINVAL;
}

// the workspace of the shortest chunk that the launch considers, which no other exceeds
static inline size_t work_len_most(const ust_grid *gr, long long wg_target) {
    GridDev g = grid_dev(gr, wg_target);
    if (g.col) {
        g.tz = column_chunk_least((long long)g.tnx * g.tny, g.nz, wg_target);
        g.tnz = (g.nz + g.tz - 1) / g.tz;
        g.ntiles = g.tnx * g.tny * g.tnz;
    }
    return work_len(g);
}

// the largest workspace any pass needs (the passes' column grids differ in z-chunk length)
extern "C" size_t ust_k_apply_work_len(const ust_grid *gr) {
    const size_t a = work_len_most(gr, UST_COL_WG_TARGET), b = work_len_most(gr, UST_COL_WG_TARGET_F32_YR);
    return a > b ? a : b;
}

extern "C" int ust_k_apply_K_cheby_prolong_f64(const ust_grid *g, const double *WK, const unsigned char *mask,
                                               double *x, const double *b, const double *invd, double *d, double c2,
                                               const double *xc, double *work, void *stream) {
    return apply_cheby_prolong<double, double>(g, WK, mask, x, x, b, invd, d, c2, xc, work, stream);
}

extern "C" int ust_k_apply_K_cheby_prolong_f32(const ust_grid *g, const float *WK, const unsigned char *mask,
                                               float *x, const float *b, const float *invd, float *d, float c2,
                                               const float *xc, float *work, void *stream) {
    return apply_cheby_prolong<float, float>(g, WK, mask, x, x, b, invd, d, c2, xc, work, stream);
}

// out of place: x before the step, xo after it (distinct vectors); on halo grids one launch, no gather
extern "C" int ust_k_apply_K_cheby_oop_f32(const ust_grid *g, const float *WK, const unsigned char *mask, const float *x,
                                           float *xo, const float *b, const float *invd, float *d, float c1, float c2,
                                           int first, float *work, void *stream) {
    if (!x || x == xo) return UST_EINVAL;
    return apply_cheby<float, float>(g, WK, mask, x, xo, b, invd, d, c1, c2, first, work, stream);
}

extern "C" int ust_k_apply_K_cheby_prolong_oop_f32(const ust_grid *g, const float *WK, const unsigned char *mask,
                                                   const float *x, float *xo, const float *b, const float *invd,
                                                   float *d, float c2, const float *xc, float *work, void *stream) {
    if (!x || x == xo) return UST_EINVAL;
    return apply_cheby_prolong<float, float>(g, WK, mask, x, xo, b, invd, d, c2, xc, work, stream);
}

extern "C" int ust_k_apply_K_f64(const ust_grid *g, const double *WK, const unsigned char *mask, const double *u,
                                 double *y, double *work, void *stream) {
    return apply_plain<double, double>(g, WK, mask, u, y, work, stream);
}

extern "C" int ust_k_apply_K_f32(const ust_grid *g, const float *WK, const unsigned char *mask, const float *u,
                                 float *y, float *work, void *stream) {
    return apply_plain<float, float>(g, WK, mask, u, y, work, stream);
}

extern "C" int ust_k_apply_K_residual_f64(const ust_grid *g, const double *WK, const unsigned char *mask,
                                          const double *u, const double *b, double *r, double *work, void *stream) {
    return apply_residual<double, double>(g, WK, mask, u, b, r, work, stream);
}

extern "C" int ust_k_apply_K_residual_f32(const ust_grid *g, const float *WK, const unsigned char *mask,
                                          const float *u, const float *b, float *r, float *work, void *stream) {
    return apply_residual<float, float>(g, WK, mask, u, b, r, work, stream);
}

extern "C" int ust_k_apply_K_cheby_f64(const ust_grid *g, const double *WK, const unsigned char *mask, double *x,
                                       const double *b, const double *invd, double *d, double c1, double c2,
                                       int first, double *work, void *stream) {
    return apply_cheby<double, double>(g, WK, mask, x, x, b, invd, d, c1, c2, first, work, stream);
}

extern "C" int ust_k_apply_K_cheby_f32(const ust_grid *g, const float *WK, const unsigned char *mask, float *x,
                                       const float *b, const float *invd, float *d, float c1, float c2, int first,
                                       float *work, void *stream) {
    return apply_cheby<float, float>(g, WK, mask, x, x, b, invd, d, c1, c2, first, work, stream);
}

// FP32 operator with bfloat16 K weights (the multigrid V-cycle's operator; half the weight stream)
extern "C" int ust_k_apply_K_f32_bf16w(const ust_grid *g, const unsigned short *WK, const unsigned char *mask,
                                       const float *u, float *y, float *work, void *stream) {
    return apply_plain<float, unsigned short>(g, WK, mask, u, y, work, stream);
}

extern "C" int ust_k_apply_K_residual_f32_bf16w(const ust_grid *g, const unsigned short *WK,
                                                const unsigned char *mask, const float *u, const float *b, float *r,
                                                float *work, void *stream) {
    return apply_residual<float, unsigned short>(g, WK, mask, u, b, r, work, stream);
}

extern "C" int ust_k_apply_K_cheby_f32_bf16w(const ust_grid *g, const unsigned short *WK, const unsigned char *mask,
                                             float *x, const float *b, const float *invd, float *d, float c1, float c2,
                                             int first, float *work, void *stream) {
    return apply_cheby<float, unsigned short>(g, WK, mask, x, x, b, invd, d, c1, c2, first, work, stream);
}

extern "C" int ust_k_apply_K_cheby_prolong_f32_bf16w(const ust_grid *g, const unsigned short *WK,
                                                     const unsigned char *mask, float *x, const float *b,
                                                     const float *invd, float *d, float c2, const float *xc,
                                                     float *work, void *stream) {
    return apply_cheby_prolong<float, unsigned short>(g, WK, mask, x, x, b, invd, d, c2, xc, work, stream);
}

extern "C" size_t ust_k_weights_len(const ust_grid *gr) {
    GridDev g = grid_dev(gr);
    if (g.dim == 3 && g.col) return (size_t)g.tnx * g.tny * g.nz * 27 * UST_TILE;
    if (g.dim == 3) return (size_t)g.ntiles * 27 * UST_TILE;
    return (size_t)g.ntiles * 9 * UST_TILE;
}

extern "C" size_t ust_k_weights_index(const ust_grid *gr, int e, int q) {
    GridDev g = grid_dev(gr);
    return widx(g, e, q);
}

// ------------------------------------------------------------------------------------------
// K u without a caller workspace, for callers that cannot allocate (code under HIP graph capture, serving
// loops): the per-tile node partials go to a file-scope device array.  Each GPU the library runs on holds its
// own copy until the process ends; its device address is looked up once per device and kept.  Every slot the
// gather pass reads is written by the same call's tile pass first, so nothing needs clearing between calls;
// calls that overlap on one GPU share the array and race.
// ------------------------------------------------------------------------------------------
#define UST_NOALLOC_WORK (size_t(1) << 22)  // doubles: 32 MiB
#define UST_NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) double scratch[UST_NOALLOC_WORK];
static double *g_scratch_dev[UST_NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_address(double **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        ust_set_hip_error(e, __FILE__, __LINE__);
        return UST_EDEVICE;
    }
    if (dev < 0 || dev >= UST_NOALLOC_MAX_DEVICES) {
        ust_set_error_text("ust_k_apply_K_f64_noalloc: device index beyond the library's table");
        return UST_EDEVICE;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            ust_set_hip_error(e != hipSuccess ? e : hipErrorInvalidSymbol, __FILE__, __LINE__);
            return UST_EDEVICE;
        }
        g_scratch_dev[dev] = (double *)p;
    }
    *out = g_scratch_dev[dev];
    return UST_OK;
}

extern "C" size_t ust_k_apply_noalloc_max_work(void) { return UST_NOALLOC_WORK; }

extern "C" int ust_k_apply_K_f64_noalloc(const ust_grid *g, const double *WK, const unsigned char *mask,
                                         const double *u, double *y, void *stream) {
    if (!g) return UST_EINVAL;
    const size_t need = work_len_most(g, col_shape(sizeof(double), EPI_Y).target);
    if (need > UST_NOALLOC_WORK) {
        char msg[256];
        snprintf(msg, sizeof(msg),
                 "ust_k_apply_K_f64_noalloc: the grid needs %zu workspace doubles, more than the %zu of the "
                 "library's static workspace (use ust_k_apply_K_f64 with a workspace)",
                 need, (size_t)UST_NOALLOC_WORK);
        ust_set_error_text(msg);
        return UST_EINVAL;
    }
    double *ws = nullptr;
    const int rc = scratch_address(&ws);
    if (rc != UST_OK) return rc;
    return apply_plain<double, double>(g, WK, mask, u, y, ws, stream);
}
