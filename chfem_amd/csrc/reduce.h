// reduce.h -- deterministic FP64 reductions shared by the kernel files:
// per-block tree sums written as block partials, summed in a fixed order by a
// separate single-block kernel (kernels.h: Reduce, Finalize,
// launch_reduce_finish).
#pragma once
#include <hip/hip_runtime.h>
#include "kernels.h"

namespace chfem {

// ---------------------------------------------------------------------------
// deterministic reductions
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// block sum; result valid in thread 0
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV])
{
    __shared__ double lds[NV][16];  // up to 1024 work-items
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double t = wave_sum(v[k]);
        if (lane == 0) lds[k][w] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double t = 0;
            for (int i = 0; i < (int)(blockDim.x + 63) / 64; i++) t += lds[k][i];
            v[k] = t;
        }
    }
    __syncthreads();
}

// a guarded launch does nothing once its Krylov loop has converged
__device__ __forceinline__ bool stopped(const Reduce &red) { return red.guard && red.S[S_DONE] != 0.0; }

// Each block writes its NV partial sums to red.partials[k * nb + block]; the
// launcher then enqueues the single-block finishing kernel, which adds the
// partials in a fixed order.  No atomics or device-scope fences: on a
// multi-XCD part a per-block release fence writes back the whole L2 of the
// XCD, and same-address atomics from thousands of blocks serialise.
template <int NV>
__device__ __forceinline__ void store_partials(const Reduce &red, double (&v)[NV])
{
    // linear block id / count: the launching grid may be 1-D, 2-D or 3-D
    const unsigned nb = gridDim.x * gridDim.y * gridDim.z;
    const unsigned bid = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    block_sum<NV>(v);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) red.partials[(size_t)k * nb + bid] = v[k];
    }
}

// Scalars of the single-kernel CG between two iterations.
struct Cg1Scalars {
    double delta, delta_old, alpha, bprev, iter, done;
};

__device__ __forceinline__ Cg1Scalars cg1_load(const double *S)
{
    return {S[S_DELTA], S[S_DELTA_OLD], S[S_ALPHA], S[S_BPREV], S[S_ITER], S[S_DONE]};
}

__device__ __forceinline__ void cg1_store(double *S, const Cg1Scalars &c)
{
    S[S_DELTA] = c.delta;
    S[S_DELTA_OLD] = c.delta_old;
    S[S_ALPHA] = c.alpha;
    S[S_BPREV] = c.bprev;
    S[S_ITER] = c.iter;
    S[S_DONE] = c.done;
}

// FIN_CG1 from the iteration's sums and the scalars it ran with (thresh < 0:
// never done)
__device__ __forceinline__ Cg1Scalars cg1_finish(double dq, double zq, double qmq, double zdz, double delta_cur,
                                                 double delta_old, double iter, double thresh)
{
    Cg1Scalars c;
    // delta of this iteration from its own z (zdz), not carried over from the
    // previous recurrence step: rounding then reaches beta through one step
    // only
    c.delta_old = zdz;
    c.alpha = zdz / dq;
    c.delta = zdz - 2.0 * c.alpha * zq + c.alpha * c.alpha * qmq;
    // the beta this iteration's launch formed its direction with (the same
    // quotient it computed), for the next launch that recovers z from the
    // directions
    c.bprev = delta_cur / delta_old;
    c.iter = iter + 1.0;
    c.done = fabs(c.delta) <= thresh ? 1.0 : 0.0;
    return c;
}

// The previous iteration's FIN_CG1 by every block of the next one (Reduce::
// prev), in the order of the finishing kernel: 4 values, 4 lists of 64 lanes
// each.  Block 0 leaves the scalars for the launch after this one.
__device__ __forceinline__ Cg1Scalars cg1_chain(const Reduce &red, unsigned nb)
{
    __shared__ double part[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (int)(blockDim.x >> 6);
    // all reads in flight before the first is used (blocks of 4 or more
    // wavefronts: up to 4 of the 16 lists each)
    double a[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int l = w + i * nw;
        const unsigned b = (l & 3) * 64 + lane;
        a[i] = l < 16 && b < nb ? red.prev[(size_t)(l >> 2) * nb + b] : 0.0;
    }
    Cg1Scalars c = cg1_load(red.Sin);
    const double thresh = red.S[S_THRESH];
#pragma unroll
    for (int i = 0; i < 4; i++) a[i] = wave_sum(a[i]);
    if (c.done == 0.0) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (lane == 0 && w + i * nw < 16) part[w + i * nw] = a[i];
        __syncthreads();
        double s[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            s[k] = 0.0;
#pragma unroll
            for (int i = 0; i < 4; i++) s[k] += part[4 * k + i];
        }
        const double alpha_at = c.iter;
        c = cg1_finish(s[0], s[1], s[2], s[3], c.delta, c.delta_old, c.iter, thresh);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            red.S[S_AHIST + (unsigned)alpha_at % S_AHIST_LEN] = c.alpha;
            red.S[S_DQ] = s[0];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) cg1_store(red.Sout, c);
    return c;
}

// element scale of a scalar density field (1 without one); same operation
// order as the reference (femhmg_thermal_3D.c:265)
__device__ __forceinline__ double sdf_scale(const Sdf &f, size_t e)
{
    return f.d ? (double)f.d[e] * (1.0 / 65535.0) * (f.fmax - f.fmin) + f.fmin : 1.0;
}

}  // namespace chfem
