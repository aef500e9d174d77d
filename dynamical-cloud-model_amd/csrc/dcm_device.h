// dcm_device.h -- device helpers shared by the kernels: index maps of the
// one-rank boundary semantics and deterministic block reductions.
#pragma once

#include "dcm_internal.h"

namespace dcm {

// Periodic source index of a lateral halo index (0 -> n, n+1 -> 1).
__device__ __forceinline__ int wrap(int j, int n) {
    return j == 0 ? n : (j == n + 1 ? 1 : j);
}
// Source level of an edge or corner on a z plane after exchange_full: the
// receive from MPI_PROC_NULL leaves the z-wrapped local copy
// (mpi_module.f90:1244-1263): 0 -> kp, kp+1 -> 1.
__device__ __forceinline__ int zwrap(int k, int kp) {
    return k == 0 ? kp : (k == kp + 1 ? 1 : k);
}
// Neumann copy of mat_ax (dynamics.f90:206-211): 0 -> 1, kp+1 -> kp.
__device__ __forceinline__ int zclamp(int k, int kp) {
    return k < 1 ? 1 : (k > kp ? kp : k);
}

// x / b by Markstein's theorem (IBM J. Res. Dev. 34, 1990): with y = 1/b
// correctly rounded, one residual step makes x*y faithful and a second one
// is the correctly rounded quotient, the IEEE one, in 5 operations instead
// of a division's dozen.  The theorem needs exact residuals: quotients near
// the ends of the exponent range take the division.  (-0 over a positive b
// gives +0, which no comparison tells from the quotient.)
__device__ __forceinline__ double div_by(double x, double b, double y) {
    const double q0 = x * y;
    const double q1 = __builtin_fma(__builtin_fma(-b, q0, x), y, q0);
    const double q2 = __builtin_fma(__builtin_fma(-b, q1, x), y, q1);
    const double ax = fabs(x);
    if (__builtin_expect(!((ax >= 0x1p-900 && ax <= 0x1p900) || x == 0.0), 0)) return x / b;
    return q2;
}
__device__ __forceinline__ float div_by(float x, float, float y) { return x * y; }
__device__ __forceinline__ double recip(double b) { return 1.0 / b; }
__device__ __forceinline__ float recip(float b) { return __builtin_amdgcn_rcpf(b); }

// Linear thread / block ids for 3-D launches.
__device__ __forceinline__ int lin_tid() {
    return threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
}
__device__ __forceinline__ unsigned lin_bid() {
    return blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
}
__device__ __forceinline__ unsigned lin_nblocks() {
    return gridDim.x * gridDim.y * gridDim.z;
}

// The sum over a wave in lane 0 by the tree of __shfl_down(v, 32), 16, ... 1:
// the same pairs, so the same bits, with the lane exchange in the VALU
// (v_permlane32_swap, v_permlane16_swap, DPP row shifts) instead of twelve
// dependent LDS permutes (measured in the fused sweeps: the block sums'
// share of a launch 3200 -> 1900 cycles).  Lanes other than 0 hold partial
// values.
template <int OFF> __device__ __forceinline__ double lane_down(double v) {
    union {
        double d;
        unsigned u[2];
    } x;
    x.d = v;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (OFF == 32)
            x.u[h] = __builtin_amdgcn_permlane32_swap(x.u[h], x.u[h], false, false)[1];
        else if (OFF == 16)
            x.u[h] = __builtin_amdgcn_permlane16_swap(x.u[h], x.u[h], false, false)[1];
        else  // row_shl:OFF
            x.u[h] = __builtin_amdgcn_update_dpp(0, x.u[h], 0x100 + OFF, 0xf, 0xf, true);
    }
    return x.d;
}
__device__ __forceinline__ double wave_sum(double v) {
    v += lane_down<32>(v);
    v += lane_down<16>(v);
    v += lane_down<8>(v);
    v += lane_down<4>(v);
    v += lane_down<2>(v);
    return v + lane_down<1>(v);
}

// the next (previous) lane's value; lane 63 (0) keeps its own
__device__ __forceinline__ double next_lane(double v) {
    union {
        double d;
        int u[2];
    } x;
    x.d = v;
#pragma unroll
    for (int h = 0; h < 2; ++h)
        x.u[h] = __builtin_amdgcn_update_dpp(x.u[h], x.u[h], 0x130, 0xf, 0xf, false);
    return x.d;
}
__device__ __forceinline__ double prev_lane(double v) {
    union {
        double d;
        int u[2];
    } x;
    x.d = v;
#pragma unroll
    for (int h = 0; h < 2; ++h)
        x.u[h] = __builtin_amdgcn_update_dpp(x.u[h], x.u[h], 0x138, 0xf, 0xf, false);
    return x.d;
}
// lane l's value in every lane (l uniform)
__device__ __forceinline__ double lane_at(double v, int l) {
    union {
        double d;
        int u[2];
    } x;
    x.d = v;
#pragma unroll
    for (int h = 0; h < 2; ++h) x.u[h] = __builtin_amdgcn_readlane(x.u[h], l);
    return x.d;
}

// Sum NS values over a block of kBlock threads in a fixed order and store
// the block's partial sums at partials[s*stride + block].  Every thread of
// the block must call this (inactive threads contribute zero).
template <int NS>
__device__ __forceinline__ void block_sum_store(double (&v)[NS], double *partials,
                                                long long stride) {
    __shared__ double red[NS][kBlock / 64];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = wave_sum(v[s]);
    const int t = lin_tid();
    const int lane = t & 63, wave = t >> 6;
    if (lane == 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) red[s][wave] = v[s];
    }
    __syncthreads();
    if (t == 0) {
        const unsigned b = lin_bid();
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double acc = red[s][0];
#pragma unroll
            for (int q = 1; q < kBlock / 64; ++q) acc += red[s][q];
            partials[s * stride + b] = acc;
        }
    }
}

// As block_sum_store, storing at partials[s*stride + idx] (idx: the block's
// tile number when blocks are renumbered).
template <int NS>
__device__ __forceinline__ void block_sum_store_at(double (&v)[NS], double *partials,
                                                   long long stride, int idx) {
    __shared__ double red[NS][kBlock / 64];
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = wave_sum(v[s]);
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    if (lane == 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) red[s][wave] = v[s];
    }
    __syncthreads();
    if (t == 0) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double acc = red[s][0];
#pragma unroll
            for (int q = 1; q < kBlock / 64; ++q) acc += red[s][q];
            partials[s * stride + idx] = acc;
        }
    }
}

__device__ __forceinline__ double block_min_store(double v, double *partials) {
    __shared__ double red[kBlock / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_down(v, off, 64);
        v = o < v ? o : v;
    }
    const int t = lin_tid();
    const int lane = t & 63, wave = t >> 6;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    if (t == 0) {
        double acc = red[0];
#pragma unroll
        for (int q = 1; q < kBlock / 64; ++q) acc = red[q] < acc ? red[q] : acc;
        partials[lin_bid()] = acc;
    }
    return v;
}

// Final reduction of one slot by a single block of 1024 threads: thread t
// sums blocks t, t+1024, ... sequentially, then a fixed tree.  Deterministic
// for a given number of blocks.
__device__ __forceinline__ double reduce_slot_1024(const double *p, int n) {
    __shared__ double red[1024];
    const int t = threadIdx.x;
    // four independent chains keep several loads in flight
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int b = t;
    for (; b + 3 * 1024 < n; b += 4 * 1024) {
        a0 += p[b];
        a1 += p[b + 1024];
        a2 += p[b + 2048];
        a3 += p[b + 3072];
    }
    for (; b < n; b += 1024) a0 += p[b];
    double acc = (a0 + a1) + (a2 + a3);
    red[t] = acc;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    double r = red[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ double reduce_min_1024(const double *p, int n) {
    __shared__ double red[1024];
    const int t = threadIdx.x;
    double acc = p[0];
    for (int b = t; b < n; b += 1024) acc = p[b] < acc ? p[b] : acc;
    red[t] = acc;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (t < w) red[t] = red[t + w] < red[t] ? red[t + w] : red[t];
        __syncthreads();
    }
    double r = red[0];
    __syncthreads();
    return r;
}

}  // namespace dcm
