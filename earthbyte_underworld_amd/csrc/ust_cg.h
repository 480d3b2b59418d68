// Device side of the inner CG's control block, shared by the vector kernels and the operator pass that forms the direction.
#ifndef UST_CG_H
#define UST_CG_H
#include "ust_common.h"

// ------------------------------------------------------------------------------------------
// The inner CG with its scalars on the device, three vector kernels per iteration and no reduction kernels between them:
// every dot product leaves one partial sum per workgroup (at most UST_CG_PARTS), and the kernel that needs the scalar
// sums them in each of its workgroups, in one fixed order, so all of them hold the same value.  A separate one-workgroup
// reduction cost a launch of 4-5 us in a chain where most kernels take 3-6 us; reading 8 KB of partials from L2 in every
// workgroup costs about 1 us, and starting a solve takes one kernel instead of six.  Whole solves with reduction kernels
// and now: 2D 64x64 FP64 136.0 -> 129.6 ms, 3D 24x16x16 FP64 699 -> 661 ms, 64x64x32 with FP32 PCG 371 -> 351 ms.
//
// Control block c: c[0] = rtol^2, c[1] = state (0 running, 1 converged, 2 NaN), c[2] = iterations taken when the state
// was last decided, c[3] = r.z of this iteration, c[4] = iterations done, c[5] = r.z of the previous one, c[6] = the
// threshold on r.r.  The direction kernel decides the state of the iterations before it: its workgroup 0 writes c[1],
// c[2], c[3] and c[6] while the others may still read them, which is safe since each workgroup decides from the same
// sums, and c[1] only changes to the state that they all find (a workgroup reading the new state stops as it would have
// done by itself).  c[4] and c[5] are written by the step kernel, which reads neither.  Once the state has left 0 both
// kernels return, so iterations launched past convergence change nothing.
// ------------------------------------------------------------------------------------------
#define CG_RZ 0
#define CG_PQ UST_CG_PARTS
#define CG_RR (2 * UST_CG_PARTS)

// sums of na partials at a and nb at b, and the control block, the same in every thread of every workgroup
struct CgSums {
    double a, b, c[7];
};
__device__ __forceinline__ CgSums cg_sums(const double *a, int na, const double *b, int nb, const double *c) {
    __shared__ double sh[8 + 7];
    double sa = 0.0, sb = 0.0;
    if (threadIdx.x < 7) sh[8 + threadIdx.x] = c[threadIdx.x];
#pragma unroll
    for (int r = 0; r < UST_CG_PARTS / 256; r++) {
        const int i = threadIdx.x + 256 * r;
        if (i < na) sa += a[i];
        if (i < nb) sb += b[i];
    }
    for (int off = 32; off > 0; off >>= 1) {
        sa += __shfl_xor(sa, off, 64);
        sb += __shfl_xor(sb, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[threadIdx.x >> 6] = sa;
        sh[4 + (threadIdx.x >> 6)] = sb;
    }
    __syncthreads();
    CgSums o;
    o.a = (sh[0] + sh[1]) + (sh[2] + sh[3]);
    o.b = (sh[4] + sh[5]) + (sh[6] + sh[7]);
    for (int k = 0; k < 7; k++) o.c[k] = sh[8 + k];
    return o;
}

// the state that the sums decide, with the threshold: before the first iteration rr is b.b
__device__ __forceinline__ double cg_state(const CgSums &s, double rr, double *thr) {
    if (s.c[1] != 0.0) return s.c[1];
    if (s.c[4] == 0.0) {
        *thr = s.c[0] * rr;
        return rr > 0.0 ? 0.0 : 1.0;
    }
    *thr = s.c[6];
    return !(rr == rr) ? 2.0 : rr <= s.c[6] ? 1.0 : 0.0;
}

#endif
