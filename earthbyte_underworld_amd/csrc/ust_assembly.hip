// PIC element assembly for gfx950: cell-sorted particles -> quadrature weights with the
// per-particle rheology fused in, and the batched B^T D B element contraction on FP64 MFMA.
//
// Reference loops restated here:
//   particle loop of _ConstitutiveMatrixCartesian_AssembleElement  ConstitutiveMatrixCartesian.c:277-410
//   rheology chain                                                   RheologyMaterial.c:240-270,
//       MaterialViscosity.c:119-131, Arrhenius.c:156-200, ViscosityLimiter.c:106-125,
//       YieldRheology.c:198-243, VonMises.c:182-269, DruckerPrager.c:236-345, TensorMath.c:430-460
//   G_e: GradientStiffnessMatrixTerm.c:220-249 ; f_e: BuoyancyForceTerm.c:370-448 ;
//   approxS_e: UzawaPreconditionerTerm.c:195-212
#include <math.h>
#include <string.h>

#include "ust_common.h"

// ------------------------------------------------------------------------------------------
// per-particle rheology (isotropic D carried as eta)
// ------------------------------------------------------------------------------------------
// per-particle yield state (strain weakening, tensile flag); pfw == nullptr: none
struct YieldDev {
    double *pfw;
    double *pfw_inc;
    unsigned char *tensile;
    double softening_strain, healing_rate;
};

// Q1 interpolation at the local coordinates xi, one axis after the other (a difference and one multiply-add per pair: a
// third of the operations of summing shape functions, and few values live at once).  v(a): the value at vertex a.
template <int DIM, typename V>
__device__ __forceinline__ double q1_value(const double *xi, V v) {
    const double fx = 0.5 * (1.0 + xi[0]), fy = 0.5 * (1.0 + xi[1]);
    double z[2] = {0.0, 0.0};
#pragma unroll
    for (int c = 0; c < (DIM == 3 ? 2 : 1); c++) {
        const double u0 = v(4 * c), u1 = v(4 * c + 1), u2 = v(4 * c + 2), u3 = v(4 * c + 3);
        const double m0 = u0 + fx * (u1 - u0), m1 = u2 + fx * (u3 - u2);
        z[c] = m0 + fy * (m1 - m0);
    }
    return DIM == 3 ? z[0] + 0.5 * (1.0 + xi[2]) * (z[1] - z[0]) : z[0];
}
// and its derivatives g along the element's axes over [0, 1]
template <int DIM, typename V>
__device__ __forceinline__ void q1_gradient(const double *xi, V v, double *g) {
    const double fx = 0.5 * (1.0 + xi[0]), fy = 0.5 * (1.0 + xi[1]);
    double gx[2] = {0.0, 0.0}, gy[2] = {0.0, 0.0}, z[2] = {0.0, 0.0};
#pragma unroll
    for (int c = 0; c < (DIM == 3 ? 2 : 1); c++) {
        const double u0 = v(4 * c), u1 = v(4 * c + 1), u2 = v(4 * c + 2), u3 = v(4 * c + 3);
        const double d0 = u1 - u0, d1 = u3 - u2, m0 = u0 + fx * d0, m1 = u2 + fx * d1;
        gx[c] = d0 + fy * (d1 - d0);
        gy[c] = m1 - m0;
        z[c] = m0 + fy * gy[c];
    }
    const double fz = DIM == 3 ? 0.5 * (1.0 + xi[2]) : 0.0;
    g[0] = DIM == 3 ? gx[0] + fz * (gx[1] - gx[0]) : gx[0];
    g[1] = DIM == 3 ? gy[0] + fz * (gy[1] - gy[0]) : gy[0];
    if (DIM == 3) g[2] = z[1] - z[0];
}

// nodal values around an element: the values of vertex a start NC doubles per node after those of its first node.  Four row
// pointers and immediate offsets: the loads need no address of their own.
template <int DIM, int NC>
struct VertexRows {
    const double *r[DIM == 3 ? 4 : 2];
    __device__ __forceinline__ VertexRows(const GridDev &g, const double *v, size_t n0) {
        r[0] = v + n0 * NC;
        r[1] = r[0] + (size_t)g.nnx * NC;
        if (DIM == 3) {
            r[2] = r[0] + (size_t)g.nnx * g.nny * NC;
            r[3] = r[2] + (size_t)g.nnx * NC;
        }
    }
    __device__ __forceinline__ double operator()(int a, int c) const { return r[a >> 1][(a & 1) * NC + c]; }
};

// what DruckerPrager takes from its friction angle: criterion = k p + 6 C cosphi f in 3D, k p + C cosphi in 2D
struct FrictionDev {
    double k, cosphi, f;
};
template <int DIM>
__device__ __forceinline__ FrictionDev friction_of(double friction) {
    const double phi = atan(friction), sinphi = sin(phi);
    FrictionDev d;
    d.cosphi = cos(phi);
    d.f = DIM == 3 ? 1.0 / (sqrt(3.0) * (3.0 - sinphi)) : 1.0;
    d.k = DIM == 3 ? 6.0 * sinphi * d.f : sinphi;
    return d;
}

// fric: friction_of the unsoftened coefficient of each of the material's rheologies
template <int DIM, bool NEED_T, bool NEED_VEL, bool SW>
__device__ double particle_viscosity(const GridDev &g, const ust_material &M, const FrictionDev *fric, size_t n0,
                                     const double *xi, const double *T, const double *vel, const double *pres, int e,
                                     float coh, int prev, const YieldDev &ys, int pi, int *yflag) {
    double eta = 0.0;
    for (int r = 0; r < M.nrh; r++) {
        const ust_rheology &rh = M.rh[r];
        if (rh.type == UST_RH_MATERIALVISCOSITY) {
            eta = rh.p[0];
        } else if (NEED_T && rh.type == UST_RH_ARRHENIUS) {
            const VertexRows<DIM, 1> tv(g, T, n0);
            const double Tp = q1_value<DIM>(xi, [&](int a) { return tv(a, 0); }), y = 0.5 * (1.0 + xi[1]);
            if (rh.p[2] > (0.0 + 1e-12)) {
                // y(xi) on a rectilinear element: ymin + (j + local fraction) * hy
                int j = (e / g.nx) % g.ny;
                double yc = g.ymin + ((double)j + y) * g.hy;
                double depth = g.ymax - yc;
                eta = rh.p[0] * exp((rh.p[1] + rh.p[2] * depth) / (Tp + rh.p[3]));
            } else {
                eta = rh.p[0] * exp((rh.p[1]) / (Tp + rh.p[3]));
            }
        } else if (rh.type == UST_RH_VISCOSITYLIMITER) {
            if (eta > rh.p[0]) eta = rh.p[0];
            if (eta < rh.p[1]) eta = rh.p[1];
        } else if (NEED_VEL && (rh.type == UST_RH_VONMISES || rh.type == UST_RH_DRUCKERPRAGER)) {
            const bool dp = rh.type == UST_RH_DRUCKERPRAGER;
            const double minVisc = dp ? rh.p[3] : rh.p[1];
            const int srSoft = (int)(dp ? rh.p[4] : rh.p[2]);
            if (!prev) continue;
            // velocity gradient at xi: L[i][k] = d u_i / d x_k
            double L[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
            const double rh3[3] = {1.0 / g.hx, 1.0 / g.hy, 1.0 / g.hz};
            const VertexRows<DIM, DIM> uv(g, vel, n0);
#pragma unroll
            for (int i = 0; i < DIM; i++) {
                q1_gradient<DIM>(xi, [&](int a) { return uv(a, i); }, L[i]);
#pragma unroll
                for (int k = 0; k < DIM; k++) L[i][k] *= rh3[k];
                // 3D: a component's 8 values at a time (all 24 at once cost a wave per SIMD)
                if (DIM == 3) asm volatile("" ::: "memory");
            }
            double inv;
            if (DIM == 3) {
                double sxx = 2.0 * eta * L[0][0], syy = 2.0 * eta * L[1][1], szz = 2.0 * eta * L[2][2];
                double sxy = eta * 2.0 * (0.5 * (L[0][1] + L[1][0]));
                double sxz = eta * 2.0 * (0.5 * (L[0][2] + L[2][0]));
                double syz = eta * 2.0 * (0.5 * (L[1][2] + L[2][1]));
                inv = 0.5 * (sxx * sxx + syy * syy + szz * szz) + sxy * sxy + sxz * sxz + syz * syz;
            } else {
                double sxx = 2.0 * eta * L[0][0], syy = 2.0 * eta * L[1][1];
                double sxy = eta * 2.0 * (0.5 * (L[0][1] + L[1][0]));
                inv = 0.5 * (sxx * sxx + syy * syy) + sxy * sxy;
            }
            double indicator = sqrt(inv);
            // strain softening of the yield parameters (VonMises.c:194-199, DruckerPrager.c:283-291): the
            // weakening state is clamped to >= 0 where it is read (StrainWeakening.c:491-492)
            const bool sw = SW && rh.p[dp ? 7 : 4] != 0.0;
            double pfw = 0.0, ratio = 0.0;
            if (sw) {
                pfw = ys.pfw[pi];
                if (pfw < 0.0) {
                    pfw = 0.0;
                    ys.pfw[pi] = 0.0;
                }
                ratio = pfw / ys.softening_strain;
                if (ratio > 1.0) ratio = 1.0;
            }
            double cohesion = (rh.p[0] * (1.0 - ratio) + rh.p[dp ? 5 : 3] * ratio) * (double)coh, criterion;
            if (!dp) {
                criterion = cohesion;
            } else {
                const FrictionDev fr = sw ? friction_of<DIM>(rh.p[1] * (1.0 - ratio) + rh.p[6] * ratio) : fric[r];
                const double c = DIM == 3 ? 6.0 * cohesion * fr.cosphi * fr.f : cohesion * fr.cosphi;
                criterion = fr.k * pres[e] + c;
                if (ys.tensile) ys.tensile[pi] = criterion <= 0.0;
                if (criterion < rh.p[2]) criterion = rh.p[2];
            }
            if (sw) {  // increment from the viscosity before yielding (StrainWeakening.c:448-482)
                const double beta = (criterion == 0.0 || indicator == 0.0) ? 0.0 : 1.0 - criterion / indicator;
                ys.pfw_inc[pi] = beta <= 0.0 ? -ys.healing_rate * pfw
                                             : (criterion / eta) * (beta / (1.0 - beta) - ys.healing_rate * pfw);
            }
            *yflag = criterion < indicator;
            if (criterion < indicator) {
                if (srSoft) {
                    eta = 2.0 * criterion * criterion * eta / (criterion * criterion + indicator * indicator);
                } else {
                    double beta = 1.0 - criterion / indicator, corr = -eta * beta;
                    if ((eta + corr) < minVisc) corr = minVisc - eta;
                    eta += corr;
                }
            }
            if (eta < minVisc) eta = minVisc;
        }
    }
    return eta;
}

// ------------------------------------------------------------------------------------------
// per-particle density of BuoyancyForceTerm_AssembleElement (BuoyancyForceTerm.c:391-425):
// rho0 (1 - alpha (T - Tref)), times (1 + beta (depth - depthref)) when beta != 0, less the background
// density of the HydrostaticTerm (HydrostaticTerm.c:267-330) at the particle's height.  full = 0: rho0.
// ------------------------------------------------------------------------------------------
struct BuoyDev {
    ust_buoyancy b;
    int full;
    double top;  // box maximum along the vertical axis
};

__device__ __forceinline__ double hydrostatic_density(const ust_buoyancy &b, double y) {
    double thick, boundary;
    if (b.hs_v != 0) {
        thick = (b.hs_height - b.hs_material_boundary) * b.hs_width / (b.hs_width + b.hs_v * b.hs_time);
        boundary = b.hs_material_boundary +
                   (b.hs_upper_density / b.hs_lower_density) * (b.hs_height - b.hs_material_boundary - thick);
    } else {
        thick = b.hs_height - b.hs_material_boundary;
        boundary = b.hs_material_boundary;
    }
    const double height = thick + boundary, h = b.hs_height - y;
    const double T = h < 0 ? b.hs_T0
                           : b.hs_T0 + b.hs_linear_coefficient * h +
                                 b.hs_exponential_coefficient1 * (1 - exp(-b.hs_exponential_coefficient2 * h));
    double density, alpha;
    if (y > height) {
        density = alpha = 0;
    } else if (y > boundary) {
        density = b.hs_upper_density;
        alpha = b.hs_upper_alpha;
    } else {
        density = b.hs_lower_density;
        alpha = b.hs_lower_alpha;
    }
    return density * (1 - alpha * T);
}

template <int DIM, bool NEED_T>
__device__ double particle_density(const GridDev &g, const BuoyDev &bd, const ust_material &M, size_t n0,
                                   const double *xi, const double *T, int e) {
    if (!bd.full) return M.density;
    const int idx[3] = {e % g.nx, (e / g.nx) % g.ny, e / (g.nx * g.ny)};
    const double mn[3] = {g.xmin, g.ymin, g.zmin}, h[3] = {g.hx, g.hy, g.hz};
    const int va = bd.b.vertical_axis;
    double cv = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++)  // no indexing by va: the arrays stay in registers
        if (d == va) cv = mn[d] + ((double)idx[d] + 0.5 * (xi[d] + 1.0)) * h[d];
    const double depth = fabs(bd.top - cv);
    double temperature = 0.0;
    if (NEED_T) {
        const VertexRows<DIM, 1> tv(g, T, n0);
        temperature = q1_value<DIM>(xi, [&](int a) { return tv(a, 0); });
    }
    double background = 0.0;
    if (bd.b.hydrostatic) background = hydrostatic_density(bd.b, mn[1] + ((double)idx[1] + 0.5 * (xi[1] + 1.0)) * h[1]);
    double density = M.density * (1.0 - M.alpha * (temperature - M.ref_temperature));
    if (M.beta != 0) density *= (1.0 + M.beta * (depth - M.ref_depth));
    return density - background;
}

// ------------------------------------------------------------------------------------------
// particles -> weights on the matrix cores.  An element's sums are products over its particles,
//   WK[qx,qy,qz] = sum_p (Lx Ly)_p[qx,qy] (w detJ eta Lz)_p[qz],   WG, WF[bx,by,bz] = sum_p (Nx Ny)_p (w detJ {1, rho} Nz)_p,
// which are exactly the four 4 x 4 blocks of v_mfma_f64_4x4x4_4b: blocks 0-2 hold the 9 x 3 products of WK, block 3 the
// 4 x 4 of WG and WF; a step takes 4 particles.  (2D: two blocks, 3 x 3 and 2 x 4, twice, so a step takes 8.)  A wave owns
// `epw` consecutive elements and reads their particles 64 at a time, one per lane: rheology, density and the 20 (2D: 12)
// factors, left in the wave's LDS (32 particles, then the other 32: LDS sets the waves in flight), where the matrix steps
// read one factor of each side per lane.  The next 64 particles are loaded while the matrix steps run.  A lane ends with
// one of the element's 43 sums, so nothing is reduced; the sums of 8 elements are written together, in 64-byte runs.
//
// The steps of the 32 staged particles add to two sums in turn, which are closed into a third where an element goes on in
// the next 32: one chain through all of an element's steps rounds once per step, which grew with the particles (rms error
// of WK against 80-bit sums, 16^3 elements: 20 particles 1.5e-16 -> 1.0e-16, 40 1.8e-16 -> 1.0e-16, 100 2.8e-16 ->
// 1.0e-16).  It costs 0 to 5% of the kernel (64^3, 40 particles per element, 231 -> 242 us; 8 particles, 112 -> 116 us);
// four sums in an unrolled loop cost 8 to 10%, closing one sum at the 32 alone was 10% less exact at 25 to 36 particles.
//
// Bound: latency, with 16 waves per CU for plain rheology (LDS) and 8 where stresses are looked up (registers: 207 in 3D).
// 21 M particles on 128x128x64, 61 materials: 842 us with lanes that accumulate the 43 sums in registers and reduce them
// through LDS, 8 waves per CU; 427 here (1.2 GB, 2.9 TB/s).  Arrhenius + DruckerPrager with cohesion noise, 4.6 M particles
// on 95x51x47: 685 -> 283 us; 3.3 M on 512x256: 228 -> 107 us (the friction terms once per material; 3 waves per SIMD for
// the 3D one, with 20 to 27 spilled registers, were slower: 437 against 392 us for the whole assembly).
//
// NEED_T / NEED_VEL / SW compile the temperature and strain-rate lookups (Arrhenius, yield) and the strain-weakening state
// in only when a material uses them.  Without them a material's chain is one number, taken once per workgroup.
// ------------------------------------------------------------------------------------------
#define PW_EPW 16
// waves wanted before a wave takes more elements: 2,048 and 32,768 measured the same within 1%
#define PW_MIN_WAVES 8192
// waves per workgroup (with lookups the material table, up to 28 KB, goes beside them into 64 KB of LDS) and the waves per
// SIMD the register budget must allow
__host__ __device__ constexpr int pw_waves(bool lookups) { return lookups ? 2 : 4; }
__host__ __device__ constexpr int pw_minb(bool lookups) { return lookups ? 2 : 4; }
__host__ __device__ constexpr int pw_factors(int dim) { return dim == 3 ? 20 : 12; }
// doubles between the rows of two particles: odd, so that the lanes' row writes spread over the LDS banks
__host__ __device__ constexpr int pw_row(int dim) { return pw_factors(dim) + 1; }
constexpr int PW_HALF = 32, PW_OUT = 8;
__host__ __device__ constexpr int pw_sums(int dim) { return dim == 3 ? 43 : 17; }
// doubles of one wave's LDS: the factors of PW_HALF particles, a row of zeros, and the sums of PW_OUT elements
__host__ __device__ constexpr int pw_wave_lds(int dim) { return (PW_HALF + 1) * pw_row(dim) + pw_sums(dim) * (PW_OUT + 1); }
// bytes of the per-workgroup material table
__host__ __device__ constexpr size_t pw_table(bool lookups, int nmat) {
    return lookups ? (size_t)nmat * (sizeof(ust_material) + UST_MAX_RHEOLOGIES * sizeof(FrictionDev))
                   : (size_t)nmat * 2 * sizeof(double);
}

struct ParticleArrays {
    const double *xi0, *xi1, *xi2, *w;
    const unsigned char *mat;
    const float *coh;
};
template <int DIM>
struct ParticleIn {
    double x[3], w;
    int m;
    float coh;
    __device__ __forceinline__ void load(const ParticleArrays &a, int p, int nmat) {
        x[0] = a.xi0[p];
        x[1] = a.xi1[p];
        x[2] = DIM == 3 ? a.xi2[p] : 0.0;
        w = a.w[p];
        m = a.mat ? (int)a.mat[p] : 0;
        m = m < nmat ? m : 0;
        coh = a.coh ? a.coh[p] : 1.0f;
    }
};

template <int DIM, bool NEED_T, bool NEED_VEL, bool SW>
__global__ __launch_bounds__(64 * pw_waves(NEED_T || NEED_VEL), pw_minb(NEED_T || NEED_VEL)) void k_particle_weights(
    GridDev g, const int *__restrict__ cell_off, ParticleArrays in, const ust_material *__restrict__ mats, int nmat,
    const double *__restrict__ T, const double *__restrict__ vel, const double *__restrict__ pres, int prev, YieldDev ys,
    BuoyDev bd, double *__restrict__ eta_out, unsigned char *__restrict__ yield_out, int epw, double *__restrict__ WK,
    double *__restrict__ WG, double *__restrict__ WF) {
    constexpr bool LOOKUPS = NEED_T || NEED_VEL;
    constexpr int PW_WAVES = pw_waves(LOOKUPS);
    constexpr int NF = pw_factors(DIM), ROW = pw_row(DIM);
    constexpr int STEP = DIM == 3 ? 4 : 8;  // particles per matrix step
    constexpr int NQ = DIM == 3 ? 27 : 9, NV = 1 << DIM, NS = pw_sums(DIM);
    extern __shared__ __align__(16) unsigned char pw_lds[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *buf = (double *)pw_lds + (size_t)wv * pw_wave_lds(DIM);
    double *osum = buf + (PW_HALF + 1) * ROW;  // osum[sum * (PW_OUT + 1) + element % PW_OUT]
    double *tab = (double *)pw_lds + (size_t)PW_WAVES * pw_wave_lds(DIM);
    // the material table: {viscosity, density}, or the materials and their friction terms
    const ust_material *smat = (const ust_material *)tab;
    const FrictionDev *sfric = (const FrictionDev *)(smat + nmat);
    if (LOOKUPS) {
        const int nw = nmat * (int)(sizeof(ust_material) / sizeof(int));
        for (int i = threadIdx.x; i < nw; i += blockDim.x) ((int *)tab)[i] = ((const int *)mats)[i];
        for (int i = threadIdx.x; i < nmat * UST_MAX_RHEOLOGIES; i += blockDim.x) {
            const ust_material &M = mats[i / UST_MAX_RHEOLOGIES];
            const int r = i % UST_MAX_RHEOLOGIES;
            FrictionDev f = {0.0, 0.0, 0.0};
            if (NEED_VEL && r < M.nrh && M.rh[r].type == UST_RH_DRUCKERPRAGER)
                f = friction_of<DIM>(M.rh[r].p[1] * (1.0 - 0.0) + M.rh[r].p[6] * 0.0);
            ((FrictionDev *)sfric)[i] = f;
        }
    } else {
        for (int i = threadIdx.x; i < nmat; i += blockDim.x) {
            int yf = -1;
            tab[2 * i] = particle_viscosity<DIM, false, false, false>(g, mats[i], nullptr, 0, nullptr, nullptr, nullptr,
                                                                       nullptr, 0, 1.0f, prev, ys, 0, &yf);
            tab[2 * i + 1] = mats[i].density;
        }
    }
    if (lane < NF) buf[PW_HALF * ROW + lane] = 0.0;
    __syncthreads();
    const int e0 = (blockIdx.x * PW_WAVES + wv) * epw;
    if (e0 >= g.nel) return;
    const int ne = min(epw, g.nel - e0);
    // lane t: the first particle of element e0 + t (t <= ne)
    const int offs = cell_off[e0 + (lane < ne ? lane : ne)];
    const int pbeg = __builtin_amdgcn_readlane(offs, 0), pend = __builtin_amdgcn_readlane(offs, ne);

    // this lane's part of a matrix step: it feeds A[i][k] and B[k][j] (i = j = lane % 4) of block b and ends with
    // D[lane / 16][lane % 4]
    const int li = lane & 3, lb = (lane >> 2) & 3, lk = lane >> 4;
    int fa, fb, sub;
    if (DIM == 3) {
        fa = lb < 3 ? min(4 * lb + li, 8) : 9 + li;
        fb = lb < 3 ? 13 + min(li, 2) : 16 + li;
        sub = lk;
    } else {
        fa = lb & 1 ? 3 + min(li, 1) : min(li, 2);
        fb = lb & 1 ? 8 + li : 5 + min(li, 2);
        sub = lk + 4 * (lb >> 1);
    }
    // which sum D is: WK's NQ, then WG's and WF's NV; -1 none
    int col = -1;
    if (DIM == 3) {
        if (lb == 3) col = NQ + (li & 2 ? NV : 0) + lk + 4 * (li & 1);
        else if (4 * lb + lk < 9 && li < 3) col = 4 * lb + lk + 9 * li;
    } else if (lb == 0) {
        if (lk < 3 && li < 3) col = lk + 3 * li;
    } else if (lb == 1 && lk < 2) {
        col = NQ + (li & 2 ? NV : 0) + lk + 2 * (li & 1);
    }
    // lane t: the slot of weight 0 of element e0 + t (t < ne <= 16)
    const unsigned long long slots = widx(g, e0 + (lane < ne ? lane : 0), 0);
    const double detJ = (DIM == 3) ? 0.125 * g.hx * g.hy * g.hz : 0.25 * g.hx * g.hy;
    double S0 = 0.0, S1 = 0.0, before = 0.0;
    int e = 0, elo = pbeg, ehi = __builtin_amdgcn_readlane(offs, 1);
    auto finish = [&]() {
        double D = (S0 + S1) + before;
        if (DIM == 2) D += __shfl_xor(D, 8);  // the two halves of a step
        if (col >= 0) osum[col * (PW_OUT + 1) + e % PW_OUT] = D;
        S0 = S1 = before = 0.0;
        e++;
        elo = ehi;
        ehi = __builtin_amdgcn_readlane(offs, e < ne ? e + 1 : ne);
        if (e % PW_OUT != 0 && e != ne) return;
        wave_sync();
        const int ef = (e - 1) / PW_OUT * PW_OUT, n = e - ef;
        const int k = lane % PW_OUT;
        const unsigned lo = __shfl((int)(unsigned)slots, ef + k), hi = __shfl((int)(slots >> 32), ef + k);
        if (k < n) {
            double *const wk = WK + (size_t)(((unsigned long long)hi << 32) | lo);
            const size_t el = (size_t)(e0 + ef + k);
#pragma unroll
            for (int t = 0; t < (NS + 64 / PW_OUT - 1) / (64 / PW_OUT); t++) {
                const int sum = lane / PW_OUT + t * (64 / PW_OUT);
                if (sum >= NS) continue;
                const double v = osum[sum * (PW_OUT + 1) + k];
                if (sum < NQ) wk[sum * UST_TILE] = v;
                else if (sum < NQ + NV) WG[(size_t)(sum - NQ) * g.nel + el] = v;
                else WF[(size_t)(sum - NQ - NV) * g.nel + el] = v;
            }
        }
        wave_sync();
    };
    ParticleIn<DIM> nxt;
    if (!LOOKUPS && pbeg < pend) nxt.load(in, min(pbeg + lane, pend - 1), nmat);
    for (int b0 = pbeg; b0 < pend; b0 += 64) {
        const int bend = min(b0 + 64, pend), p = min(b0 + lane, pend - 1);
        ParticleIn<DIM> q = nxt;
        if (LOOKUPS) q.load(in, p, nmat);  // the registers of a load ahead would cost a wave
        else if (bend < pend) nxt.load(in, min(bend + lane, pend - 1), nmat);
        // lanes past the last particle repeat it; their rows are not read
        double eta, rho;
        const ust_material &M = LOOKUPS ? smat[q.m] : mats[q.m];
        if (LOOKUPS || bd.full) {
            int pe = 0;
            for (int t = 1; t < ne; t++) pe += p >= __builtin_amdgcn_readlane(offs, t);
            pe += e0;
            const int ie = pe % g.nx, je = (pe / g.nx) % g.ny, ke = pe / (g.nx * g.ny);
            const size_t n0 = (size_t)ie + (size_t)g.nnx * ((size_t)je + (size_t)g.nny * ke);  // the element's first node
            int yf = -1;
            if (LOOKUPS) {
                eta = particle_viscosity<DIM, NEED_T, NEED_VEL, SW>(g, M, sfric + q.m * UST_MAX_RHEOLOGIES, n0, q.x, T,
                                                                    vel, pres, pe, q.coh, prev, ys, p, &yf);
                if (NEED_VEL && yield_out && yf >= 0) yield_out[p] = (unsigned char)yf;
            } else {
                eta = tab[2 * q.m];
            }
            rho = particle_density<DIM, NEED_T>(g, bd, M, n0, q.x, T, pe);
        } else {
            eta = tab[2 * q.m];
            rho = tab[2 * q.m + 1];
        }
        if (eta_out) eta_out[p] = eta;
        const double wd = q.w * detJ, et = wd * eta, wr = wd * rho;
        for (int h0 = b0; h0 < bend; h0 += PW_HALF) {
            const int hend = min(h0 + PW_HALF, bend);
            if (lane / PW_HALF == (h0 - b0) / PW_HALF) {
                double *r = buf + (lane % PW_HALF) * ROW;
                // taken anew in each half: the factors, hoisted out of the loop, would hold 40 registers through it
                double x0 = q.x[0], x1 = q.x[1], x2 = q.x[2];
                asm volatile("" : "+v"(x0), "+v"(x1), "+v"(x2));
                double Lx[3], Ly[3], Lz[3];
                lagrange3(x0, Lx);
                lagrange3(x1, Ly);
                if (DIM == 3) lagrange3(x2, Lz);
                const double Nx[2] = {0.5 * (1.0 - x0), 0.5 * (1.0 + x0)};
                const double Ny[2] = {0.5 * (1.0 - x1), 0.5 * (1.0 + x1)};
                const double Nz[2] = {0.5 * (1.0 - x2), 0.5 * (1.0 + x2)};
                if (DIM == 3) {
#pragma unroll
                    for (int t = 0; t < 9; t++) r[t] = Lx[t % 3] * Ly[t / 3];
#pragma unroll
                    for (int t = 0; t < 4; t++) r[9 + t] = Nx[t & 1] * Ny[t >> 1];
#pragma unroll
                    for (int t = 0; t < 3; t++) r[13 + t] = et * Lz[t];
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        r[16 + t] = wd * Nz[t];
                        r[18 + t] = wr * Nz[t];
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < 3; t++) {
                        r[t] = Lx[t];
                        r[5 + t] = et * Ly[t];
                    }
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        r[3 + t] = Nx[t];
                        r[8 + t] = wd * Ny[t];
                        r[10 + t] = wr * Ny[t];
                    }
                }
            }
            wave_sync();
            while (e < ne) {
                const int lo = max(elo, h0) - h0, hi = min(ehi, hend) - h0;
                if (lo < hi) {  // the next step's factors are read while this one multiplies
                    int row = lo + sub < hi ? lo + sub : PW_HALF;
                    double a = buf[row * ROW + fa], b = buf[row * ROW + fb];
                    for (int st = lo + STEP; st < hi; st += STEP) {
                        row = st + sub < hi ? st + sub : PW_HALF;
                        const double an = buf[row * ROW + fa], bn = buf[row * ROW + fb];
                        const double t = S1 + __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, 0.0, 0, 0, 0);
                        S1 = S0;
                        S0 = t;
                        a = an;
                        b = bn;
                    }
                    S1 += __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, 0.0, 0, 0, 0);
                }
                if (ehi > hend) {  // the element goes on in the next particles
                    before += S0 + S1;
                    S0 = S1 = 0.0;
                    break;
                }
                finish();
            }
            wave_sync();
        }
    }
    while (e < ne) finish();  // elements without particles
}

// ------------------------------------------------------------------------------------------
// B(xi_q)^T D0 B(xi_q) entry (row (a,i), col (b,j)) on the Lagrange point q, from the global
// shape-function derivatives GNx_k(a) at q:  delta_ij sum_k GNx_k(a) GNx_k(b) + GNx_j(a) GNx_i(b)
// ------------------------------------------------------------------------------------------
template <int DIM>
__device__ __forceinline__ double gnx_at(int a, int k, int q, const double *s) {
    // s_k * dN_a/dxi_k at Lagrange point q:  sgn(a_k) prod_{d != k} cfac(a_d, q_d) / 2^DIM
    int qd[3] = {q % 3, (q / 3) % 3, q / 9};
    int v = sgn((a >> k) & 1);
#pragma unroll
    for (int d = 0; d < DIM; d++)
        if (d != k) v *= cfac((a >> d) & 1, qd[d]);
    return s[k] * (double)v / (double)(1 << DIM);
}

typedef double ust_double4 __attribute__((ext_vector_type(4)));

// K_e = W (count x NQ) * M (NQ x nd^2) on v_mfma_f64_16x16x4f64.  One wavefront per 16 elements;
// A fragment: lane l holds A[l%16][l/16], B fragment: B[l/16][l%16], D: acc[r] = D[4r + l/16][l%16]
// (output layout measured on gfx950 against the oracle's element matrices).  The B operand M[q][(a,i),(b,j)]
// is built from the shape-function derivatives at the Lagrange points, GN[a][k][q] (2^DIM x DIM x NQ values),
// which the workgroup tabulates in LDS once: an entry of M is then at most four products of table values.
template <int DIM>
__global__ __launch_bounds__(256) void k_element_matrices(GridDev g, const double *__restrict__ WK, int first,
                                                          int count, double *__restrict__ Ke) {
    constexpr int NQ = DIM == 3 ? 27 : 9;
    constexpr int NV = 1 << DIM;
    constexpr int ND = NV * DIM;
    constexpr int NCOL = ND * ND;
    constexpr int KSTEPS = (NQ + 3) / 4;
    constexpr int NG = NV * DIM * NQ;
    __shared__ double gn[NG];  // gn[(a*DIM + k)*NQ + q]
    const double s[3] = {2.0 / g.hx, 2.0 / g.hy, 2.0 / g.hz};
    for (int t = threadIdx.x; t < NG; t += blockDim.x) {
        const int q = t % NQ, ak = t / NQ;
        gn[t] = gnx_at<DIM>(ak / DIM, ak % DIM, q, s);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int e0 = tile * 16;
    if (e0 >= count) return;
    const int li = lane & 15, lk = lane >> 4;
    double afrag[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
        const int q = ks * 4 + lk, el = e0 + li;
        afrag[ks] = (q < NQ && el < count) ? WK[widx(g, first + el, q)] : 0.0;
    }
    for (int ct = 0; ct < NCOL / 16; ct++) {
        ust_double4 acc = {0.0, 0.0, 0.0, 0.0};
        const int col = ct * 16 + li;
        const int row = col / ND, cin = col % ND;
        const int a = row / DIM, i = row % DIM, b = cin / DIM, j = cin % DIM;
        const double *ga = gn + a * DIM * NQ, *gb = gn + b * DIM * NQ;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) {
            const int q = ks * 4 + lk;
            double m = 0.0;
            if (q < NQ) {
                if (i == j) {
#pragma unroll
                    for (int k = 0; k < DIM; k++) m += ga[k * NQ + q] * gb[k * NQ + q];
                }
                m += ga[j * NQ + q] * gb[i * NQ + q];
            }
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(afrag[ks], m, acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int el = e0 + 4 * r + lk;
            if (el < count) Ke[(size_t)el * NCOL + col] = acc[r];
        }
    }
}

// G_e[a,i] = -(sgn(a_i)/h_i) (WG[b_i=0,b_perp=a_perp] + WG[b_i=1,b_perp=a_perp])
template <int DIM>
__device__ __forceinline__ void element_G(const GridDev &g, const double *WG, int e, double *Ge) {
    constexpr int NV = 1 << DIM;
    double wv[NV];
#pragma unroll
    for (int b = 0; b < NV; b++) wv[b] = WG[(size_t)b * g.nel + e];
    const double h[3] = {g.hx, g.hy, g.hz};
#pragma unroll
    for (int a = 0; a < NV; a++)
#pragma unroll
        for (int i = 0; i < DIM; i++) {
            const int b0 = a & ~(1 << i), b1 = a | (1 << i);
            Ge[a * DIM + i] = -(double)sgn((a >> i) & 1) / h[i] * (wv[b0] + wv[b1]);
        }
}

template <int DIM>
__global__ void k_element_G(GridDev g, const double *__restrict__ WG, int first, int count, double *__restrict__ Ge) {
    constexpr int ND = (1 << DIM) * DIM;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    double ge[ND];
    element_G<DIM>(g, WG, first + t, ge);
#pragma unroll
    for (int v = 0; v < ND; v++) Ge[(size_t)t * ND + v] = ge[v];
}

struct FDir {
    double d[3];
};

template <int DIM>
__global__ void k_element_f(GridDev g, const double *__restrict__ WF, double gravity, FDir dir, int first, int count,
                            double *__restrict__ fe) {
    constexpr int NV = 1 << DIM, ND = NV * DIM;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
#pragma unroll
    for (int a = 0; a < NV; a++)
#pragma unroll
        for (int i = 0; i < DIM; i++)
            fe[(size_t)t * ND + a * DIM + i] = dir.d[i] != 0.0 ? gravity * dir.d[i] * WF[(size_t)a * g.nel + first + t]
                                                                : 0.0;
}

// BuoyancyForceTerm "adjust": WF *= 2^dim detJ / sum_b WG[b] (= 2^dim / the element's sum of weights)
template <int DIM>
__global__ void k_adjust_force(GridDev g, const double *__restrict__ WG, double *__restrict__ WF) {
    constexpr int NV = 1 << DIM;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const double detJ = (DIM == 3) ? 0.125 * g.hx * g.hy * g.hz : 0.25 * g.hx * g.hy;
    double s = 0.0;
#pragma unroll
    for (int b = 0; b < NV; b++) s += WG[(size_t)b * g.nel + e];
    const double f = s > 0.0 ? (double)NV * detJ / s : 1.0;
#pragma unroll
    for (int b = 0; b < NV; b++) WF[(size_t)b * g.nel + e] *= f;
}

// diag of K_e: sum_q W_q (sum_k GNx_k(a)^2 + GNx_i(a)^2), with GNx_k(a)^2 = s_k^2 / 4^DIM prod_{d != k} cfac^2.  Per
// direction k the weights are summed along k, then taken against cfac^2 = {4, 1, 0} or {0, 1, 4} along the others.
template <int DIM>
__device__ __forceinline__ void element_K_diag(const GridDev &g, const double *__restrict__ WK, int e, double *dg) {
    constexpr int NQ = DIM == 3 ? 27 : 9, NV = 1 << DIM;
    const double s[3] = {2.0 / g.hx, 2.0 / g.hy, 2.0 / g.hz};
    const double *w = WK + widx(g, e, 0);
    double W[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) W[q] = w[q * UST_TILE];
#pragma unroll
    for (int v = 0; v < NV * DIM; v++) dg[v] = 0.0;
#pragma unroll
    for (int k = 0; k < DIM; k++) {
        constexpr int p3[3] = {1, 3, 9};
        const int u = k == 0 ? 1 : 0, v = k == 2 ? 1 : 2;  // the other axes (v: 3D only)
        const double t = s[k] * s[k] / (double)(1 << (2 * DIM));
        double c[2][3];  // [bit on u][point on v]
#pragma unroll
        for (int qv = 0; qv < (DIM == 3 ? 3 : 1); qv++) {
            double l[3];
#pragma unroll
            for (int qu = 0; qu < 3; qu++) {
                const int i = qu * p3[u] + (DIM == 3 ? qv * p3[v] : 0);
                l[qu] = W[i] + W[i + p3[k]] + W[i + 2 * p3[k]];
            }
            c[0][qv] = 4.0 * l[0] + l[1];
            c[1][qv] = l[1] + 4.0 * l[2];
        }
#pragma unroll
        for (int a = 0; a < NV; a++) {
            const double *cu = c[(a >> u) & 1];
            const double d = t * (DIM == 3 ? ((a >> v) & 1 ? cu[1] + 4.0 * cu[2] : 4.0 * cu[0] + cu[1]) : cu[0]);
#pragma unroll
            for (int i = 0; i < DIM; i++) dg[a * DIM + i] += i == k ? 2.0 * d : d;
        }
    }
}

// approxS = g^T diag(K_e)^-1 g (UzawaPreconditionerTerm.c:195-212)
template <int DIM>
__device__ __forceinline__ double uzawa_diag(const GridDev &g, const double *__restrict__ WK,
                                             const double *__restrict__ WG, int e, double *ge) {
    constexpr int ND = (1 << DIM) * DIM;
    double dg[ND];
    element_K_diag<DIM>(g, WK, e, dg);
    element_G<DIM>(g, WG, e, ge);
    double s = 0.0;
#pragma unroll
    for (int v = 0; v < ND; v++) s += ge[v] * (ge[v] / dg[v]);
    return s;
}

template <int DIM>
__global__ __launch_bounds__(256, 4) void k_uzawa_diag(GridDev g, const double *__restrict__ WK,
                                                    const double *__restrict__ WG, double *__restrict__ approxS) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    double ge[(1 << DIM) * DIM];
    approxS[e] = uzawa_diag<DIM>(g, WK, WG, e, ge);
}

// ------------------------------------------------------------------------------------------
// What an assembly derives from the weights, in one pass over the elements and one over the nodes, with the two norms of
// the null-space test on the way (ksp_pressure_nullspace.c:139-158): a third launch leaves them in host memory.  Before,
// thirteen launches and two copies with a wait each: 45 of the 72 us of a 64x64 assembly, 270 of 671 us at 128x128x64.
// ------------------------------------------------------------------------------------------
constexpr int DERIVE_BLOCKS = 1024;  // partial results per pass

// approxS, h = 0 and per block the largest row sum of |D| over the free dofs
template <int DIM>
__global__ __launch_bounds__(256, 4) void k_derive_elements(GridDev g, const double *__restrict__ WK,
                                                         const double *__restrict__ WG,
                                                         const unsigned char *__restrict__ mask,
                                                         double *__restrict__ approxS, double *__restrict__ h,
                                                         double *__restrict__ partial) {
    constexpr int NV = 1 << DIM;
    __shared__ double sh[4];
    double m = 0.0;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < g.nel; e += gridDim.x * 256) {
        const int ex = e % g.nx, ey = (e / g.nx) % g.ny, ez = e / (g.nx * g.ny);
        const unsigned char *mk = mask + ((size_t)ex + (size_t)g.nnx * ((size_t)ey + (size_t)g.nny * ez)) * DIM;
        unsigned char bc[NV * DIM];
#pragma unroll
        for (int a = 0; a < NV; a++)
#pragma unroll
            for (int i = 0; i < DIM; i++)
                bc[a * DIM + i] = mk[((size_t)(a & 1) + (size_t)g.nnx * ((a >> 1) & 1) +
                                      (DIM == 3 ? (size_t)g.nnx * g.nny * (a >> 2) : 0)) * DIM + i];
        double ge[NV * DIM];
        approxS[e] = uzawa_diag<DIM>(g, WK, WG, e, ge);
        h[e] = 0.0;
        double s = 0.0;
#pragma unroll
        for (int v = 0; v < NV * DIM; v++) s += bc[v] ? 0.0 : fabs(ge[v]);
        m = fmax(m, s);
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
}

// f = gravity dir sum of WF around the node (0 on Dirichlet dofs) and per block the sum of squares of G 1
template <int DIM>
__global__ __launch_bounds__(256) void k_derive_nodes(GridDev g, const double *__restrict__ WG,
                                                      const double *__restrict__ WF, double gravity, FDir dir,
                                                      const unsigned char *__restrict__ mask, double *__restrict__ f,
                                                      double *__restrict__ partial) {
    constexpr int NV = 1 << DIM;
    __shared__ double sh[4];
    const double hr[3] = {1.0 / g.hx, 1.0 / g.hy, 1.0 / g.hz};
    const int nnodes = g.nnx * g.nny * g.nnz;
    double s = 0.0;
    for (int n = blockIdx.x * 256 + threadIdx.x; n < nnodes; n += gridDim.x * 256) {
        const int gx = n % g.nnx, gy = (n / g.nnx) % g.nny, gz = n / (g.nnx * g.nny);
        double fn = 0.0, gn[DIM];
#pragma unroll
        for (int i = 0; i < DIM; i++) gn[i] = 0.0;
#pragma unroll
        for (int a = 0; a < NV; a++) {
            const int ex = gx - (a & 1), ey = gy - ((a >> 1) & 1), ez = DIM == 3 ? gz - (a >> 2) : 0;
            const bool in = ex >= 0 && ey >= 0 && ez >= 0 && ex < g.nx && ey < g.ny && ez < g.nz;
            const size_t e = in ? (size_t)ex + (size_t)g.nx * ((size_t)ey + (size_t)g.ny * ez) : 0;
            const double wa = WG[(size_t)a * g.nel + e], wf = WF[(size_t)a * g.nel + e];
            double wi[DIM];
#pragma unroll
            for (int i = 0; i < DIM; i++) wi[i] = WG[(size_t)(a ^ (1 << i)) * g.nel + e];
            if (!in) continue;
            fn += wf;
#pragma unroll
            for (int i = 0; i < DIM; i++) gn[i] -= (double)sgn((a >> i) & 1) * hr[i] * (wa + wi[i]);
        }
#pragma unroll
        for (int i = 0; i < DIM; i++) {
            const size_t dof = (size_t)n * DIM + i;
            const bool bc = mask[dof] != 0;
            f[dof] = bc || dir.d[i] == 0.0 ? 0.0 : gravity * dir.d[i] * fn;
            s += bc ? 0.0 : gn[i] * gn[i];
        }
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// out[0] = the sum of the first ns partials, out[1] = the largest of the nm at DERIVE_BLOCKS
__global__ __launch_bounds__(256) void k_derive_norms(const double *__restrict__ partial, int ns, int nm,
                                                      double *__restrict__ out) {
    __shared__ double sh[2][4];
    double s = 0.0, m = 0.0;
    for (int i = threadIdx.x; i < ns; i += 256) s += partial[i];
    for (int i = threadIdx.x; i < nm; i += 256) m = fmax(m, partial[DERIVE_BLOCKS + i]);
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_xor(s, off, 64);
        m = fmax(m, __shfl_xor(m, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = s;
        sh[1][threadIdx.x >> 6] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
        out[1] = fmax(fmax(sh[1][0], sh[1][1]), fmax(sh[1][2], sh[1][3]));
    }
}

// ------------------------------------------------------------------------------------------
extern "C" int ust_k_particle_weights(const ust_grid *gr, const int *cell_off, int ppc_hint, const double *xi0,
                                      const double *xi1, const double *xi2, const double *w,
                                      const unsigned char *mat, const float *coh_scale,
                                      const ust_material *materials_dev, int nmat, const double *temperature,
                                      const double *velocity, const double *pressure, int prev_solution,
                                      const ust_yield_state *yield_state, const ust_buoyancy *buoyancy,
                                      double *eta_out, unsigned char *yield_out, double *WK, double *WG, double *WF,
                                      void *stream) {
    if (!gr || !cell_off || !xi0 || !xi1 || !w || !materials_dev || !WK || !WG || !WF) return UST_EINVAL;
    if (gr->dim == 3 && !xi2) return UST_EINVAL;
    if (nmat < 1 || nmat > UST_MAX_MATERIALS) return UST_EINVAL;
    GridDev g = grid_dev(gr);
    if (g.nel <= 0) return UST_OK;
    BuoyDev bd;
    memset(&bd, 0, sizeof(bd));
    if (buoyancy) {
        if (buoyancy->vertical_axis < 0 || buoyancy->vertical_axis >= gr->dim) return UST_EINVAL;
        bd.b = *buoyancy;
        bd.full = 1;
        bd.top = gr->xmax[buoyancy->vertical_axis];
    }
    YieldDev ys = {nullptr, nullptr, nullptr, 1.0, 0.0};
    if (yield_state) {
        if (yield_state->pfw && (!yield_state->pfw_inc || !(yield_state->softening_strain > 0.0))) return UST_EINVAL;
        ys.pfw = yield_state->pfw;
        ys.pfw_inc = yield_state->pfw_inc;
        ys.tensile = yield_state->tensile;
        ys.softening_strain = yield_state->softening_strain;
        ys.healing_rate = yield_state->healing_rate;
    }
    // temperature / velocity lookups only when a rheology or the density reads them (the caller passes NULL
    // otherwise)
    const bool needT = temperature != nullptr, needV = velocity != nullptr && pressure != nullptr;
    hipStream_t st = ust_stream(stream);
    (void)ppc_hint;
    // elements per wave: 16 (a row of a weight tile, whose stores fill cache lines) once that leaves enough waves to fill
    // the GPU several times over, fewer on smaller grids
    int epw = PW_EPW;
    while (epw > 1 && g.nel / epw < PW_MIN_WAVES) epw /= 2;
    const int waves = pw_waves(needT || needV);
    const unsigned grid = ust_grid_size((size_t)g.nel, waves * epw);
    const bool sw = needV && ys.pfw != nullptr;  // compiled in only when the yield state carries it (it costs registers)
    const ParticleArrays in = {xi0, xi1, xi2, w, mat, coh_scale};
    const size_t lds = (size_t)waves * pw_wave_lds(g.dim) * sizeof(double) + pw_table(needT || needV, nmat);
#define LAUNCH_PW(D, NT, NVL, SWK)                                                                                      \
    hipLaunchKernelGGL((k_particle_weights<D, NT, NVL, SWK>), dim3(grid), dim3(64 * waves), lds, st, g, cell_off, in, \
                       materials_dev, nmat, temperature, velocity, pressure, prev_solution, ys, bd, eta_out, yield_out,  \
                       epw, WK, WG, WF)
#define LAUNCH_F(D)                                              \
    do {                                                         \
        if (needT && needV && sw) LAUNCH_PW(D, true, true, true); \
        else if (needT && needV) LAUNCH_PW(D, true, true, false); \
        else if (needT) LAUNCH_PW(D, true, false, false);         \
        else if (needV && sw) LAUNCH_PW(D, false, true, true);    \
        else if (needV) LAUNCH_PW(D, false, true, false);         \
        else LAUNCH_PW(D, false, false, false);                   \
    } while (0)
    if (g.dim == 3) LAUNCH_F(3);
    else LAUNCH_F(2);
#undef LAUNCH_F
#undef LAUNCH_PW
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_element_matrices(const ust_grid *gr, const double *WK, int first, int count, double *Ke,
                                      void *stream) {
    GridDev g = grid_dev(gr);
    if (first < 0 || count < 0 || first + count > g.nel || !WK || !Ke) return UST_EINVAL;
    if (count == 0) return UST_OK;
    const int tiles = (count + 15) / 16;
    const unsigned grid = ust_grid_size(tiles, UST_BLOCK / 64);
    if (g.dim == 3)
        hipLaunchKernelGGL(k_element_matrices<3>, dim3(grid), dim3(UST_BLOCK), 0, ust_stream(stream), g, WK, first,
                           count, Ke);
    else
        hipLaunchKernelGGL(k_element_matrices<2>, dim3(grid), dim3(UST_BLOCK), 0, ust_stream(stream), g, WK, first,
                           count, Ke);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_element_G(const ust_grid *gr, const double *WG, int first, int count, double *Ge,
                               void *stream) {
    GridDev g = grid_dev(gr);
    if (first < 0 || count < 0 || first + count > g.nel || !WG || !Ge) return UST_EINVAL;
    if (count == 0) return UST_OK;
    if (g.dim == 3)
        hipLaunchKernelGGL(k_element_G<3>, dim3(ust_grid_size(count, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WG, first, count, Ge);
    else
        hipLaunchKernelGGL(k_element_G<2>, dim3(ust_grid_size(count, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WG, first, count, Ge);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_element_f_dir(const ust_grid *gr, const double *WF, double gravity, const double *dir,
                                   int first, int count, double *fe, void *stream) {
    GridDev g = grid_dev(gr);
    if (first < 0 || count < 0 || first + count > g.nel || !WF || !fe || !dir) return UST_EINVAL;
    if (count == 0) return UST_OK;
    FDir d = {{dir[0], dir[1], g.dim == 3 ? dir[2] : 0.0}};
    if (g.dim == 3)
        hipLaunchKernelGGL(k_element_f<3>, dim3(ust_grid_size(count, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WF, gravity, d, first, count, fe);
    else
        hipLaunchKernelGGL(k_element_f<2>, dim3(ust_grid_size(count, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WF, gravity, d, first, count, fe);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_element_f(const ust_grid *gr, const double *WF, double gravity, int first, int count,
                               double *fe, void *stream) {
    const double down[3] = {0.0, -1.0, 0.0};
    return ust_k_element_f_dir(gr, WF, gravity, down, first, count, fe, stream);
}

extern "C" int ust_k_adjust_force_weights(const ust_grid *gr, const double *WG, double *WF, void *stream) {
    GridDev g = grid_dev(gr);
    if (!WG || !WF) return UST_EINVAL;
    if (g.nel == 0) return UST_OK;
    if (g.dim == 3)
        hipLaunchKernelGGL(k_adjust_force<3>, dim3(ust_grid_size(g.nel, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WG, WF);
    else
        hipLaunchKernelGGL(k_adjust_force<2>, dim3(ust_grid_size(g.nel, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WG, WF);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_uzawa_diag(const ust_grid *gr, const double *WK, const double *WG, double *approxS,
                                void *stream) {
    GridDev g = grid_dev(gr);
    if (!WK || !WG || !approxS) return UST_EINVAL;
    if (g.dim == 3)
        hipLaunchKernelGGL(k_uzawa_diag<3>, dim3(ust_grid_size(g.nel, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WK, WG, approxS);
    else
        hipLaunchKernelGGL(k_uzawa_diag<2>, dim3(ust_grid_size(g.nel, UST_BLOCK)), dim3(UST_BLOCK), 0,
                           ust_stream(stream), g, WK, WG, approxS);
    UST_LAUNCH_CHECK();
    return UST_OK;
}

extern "C" int ust_k_derive(const ust_grid *gr, const double *WK, const double *WG, const double *WF, double gravity,
                            const double *dir, const unsigned char *mask, double *approxS, double *f, double *h,
                            double *partial, double *norms, void *stream) {
    if (!gr || !WK || !WG || !WF || !dir || !mask || !approxS || !f || !h || !partial || !norms) return UST_EINVAL;
    GridDev g = grid_dev(gr);
    if (g.nel <= 0) return UST_EINVAL;
    const FDir d = {{dir[0], dir[1], g.dim == 3 ? dir[2] : 0.0}};
    hipStream_t st = ust_stream(stream);
    const unsigned be = ust_grid_size((size_t)g.nel, 256), bn = ust_grid_size((size_t)g.nnx * g.nny * g.nnz, 256);
    const int ne = (int)(be < DERIVE_BLOCKS ? be : DERIVE_BLOCKS), nn = (int)(bn < DERIVE_BLOCKS ? bn : DERIVE_BLOCKS);
    if (g.dim == 3) {
        hipLaunchKernelGGL(k_derive_elements<3>, dim3(ne), dim3(256), 0, st, g, WK, WG, mask, approxS, h,
                           partial + DERIVE_BLOCKS);
        hipLaunchKernelGGL(k_derive_nodes<3>, dim3(nn), dim3(256), 0, st, g, WG, WF, gravity, d, mask, f, partial);
    } else {
        hipLaunchKernelGGL(k_derive_elements<2>, dim3(ne), dim3(256), 0, st, g, WK, WG, mask, approxS, h,
                           partial + DERIVE_BLOCKS);
        hipLaunchKernelGGL(k_derive_nodes<2>, dim3(nn), dim3(256), 0, st, g, WG, WF, gravity, d, mask, f, partial);
    }
    hipLaunchKernelGGL(k_derive_norms, dim3(1), dim3(256), 0, st, partial, nn, ne, norms);
    UST_LAUNCH_CHECK();
    return UST_OK;
}
