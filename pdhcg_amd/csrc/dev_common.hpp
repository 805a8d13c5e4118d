// Device-side building blocks for gfx950 (CDNA4, wave64): error checking,
// wave/block reductions and a deterministic grid reduction.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "host_common.h"

#define HIP_OK(call)                                                                                   \
    do {                                                                                               \
        hipError_t err_ = (call);                                                                      \
        if (err_ != hipSuccess)                                                                        \
            ::pdhcg::fail("HIP error %s at %s:%d: %s", hipGetErrorName(err_), __FILE__, __LINE__,      \
                          hipGetErrorString(err_));                                                    \
    } while (0)

namespace pdhcg {

constexpr int kWave = 64;
constexpr int kBlock = 256;            // threads per block of the elementwise/reduction kernels
constexpr int kMaxRedBlocks = 4096;    // upper bound on blocks of any reducing launch
constexpr int kMaxRedValues = 16;      // values reduced by one launch
constexpr size_t kRedPartials = (size_t)kMaxRedValues * kMaxRedBlocks;

template <class T> __device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Sum over `width` consecutive lanes (width a power of two <= 64); every lane
// of the group receives the group total.
template <class T> __device__ __forceinline__ T group_sum(T v, int width) {
    for (int off = width >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Cross-lane moves in the vector ALU: a DPP move, or the exchange of halves
// and rows that gfx950 has as v_permlane32_swap / v_permlane16_swap.  A wave
// total takes about 150 cycles this way, 800 through ds_bpermute (__shfl_xor).
template <int Ctrl> __device__ __forceinline__ double dpp_move(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, Ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), Ctrl, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E;                // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kDppHalfMirror = 0x141, kDppMirror = 0x140;      // lane i -> 7 - i of 8, 15 - i of 16
constexpr int kDppRor8 = 0x128;                                // lane i -> i xor 8 of 16

// a's total over lanes l and l xor 32 in the lower half, b's in the upper half.
__device__ __forceinline__ double fold32(double a, double b) {
    const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
// The same over lanes l and l xor 16: a's in the even rows of 16, b's in the odd rows.
__device__ __forceinline__ double fold16(double a, double b) {
    const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
// Total over 16 lanes, and over the wave, in every lane.
__device__ __forceinline__ double row_total(double v) {
    v += dpp_move<kDppXor1>(v);
    v += dpp_move<kDppXor2>(v);
    v += dpp_move<kDppHalfMirror>(v);
    return v + dpp_move<kDppMirror>(v);
}
__device__ __forceinline__ double wave_total(double v) {
    v = row_total(v);
    v = fold16(v, v);
    return fold32(v, v);
}

// Total over L consecutive lanes (a power of two), in every lane of the group.
template <int L> __device__ __forceinline__ double group_total(double v) {
    if (L >= 2) v += dpp_move<kDppXor1>(v);
    if (L >= 4) v += dpp_move<kDppXor2>(v);
    if (L >= 8) v += dpp_move<kDppHalfMirror>(v);
    if (L >= 16) v += dpp_move<kDppMirror>(v);
    if (L >= 32) v = fold16(v, v);
    if (L >= 64) v = fold32(v, v);
    return v;
}

// Combines two partial values: the first NS of a value pack are sums, the
// remaining ones are maxima.
template <int NS> __device__ __forceinline__ double combine(int i, double a, double b) {
    return i < NS ? a + b : fmax(a, b);
}

// Reduction request: the output receives NS sums followed by NM maxima (FP64).
// A reducing kernel writes one partial pack per workgroup; the fold kernel
// launched after it on the same stream combines them (no atomics, no fences:
// the kernel boundary orders the writes before the reads).
struct GridRed {
    double *partials;   // kRedPartials: [kMaxRedValues][kMaxRedBlocks]
    double *out;
};

// Load of a value written by another workgroup of the same launch: coherent
// at device scope (bypasses a possibly stale per-CU cache line) but, unlike a
// volatile access, free to be pipelined with other loads.
__device__ __forceinline__ double coherent_load(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Block reduction of a value pack into thread 0 (fixed combination order).
template <int NS, int NM> __device__ __forceinline__ void block_reduce(double (&v)[NS + NM], double *lds) {
    constexpr int NV = NS + NM;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, waves = blockDim.x / kWave;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) v[i] = combine<NS>(i, v[i], __shfl_xor(v[i], off, kWave));
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) lds[i * 16 + wave] = v[i];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double a = lds[i * 16];
            for (int w = 1; w < waves; ++w) a = combine<NS>(i, a, lds[i * 16 + w]);
            v[i] = a;
        }
    __syncthreads();
}

// Stores this workgroup's partial pack (thread 0 writes after a block
// reduction in a fixed order).  Launch grid_fold_kernel with the same grid
// size afterwards.
template <int NS, int NM> __device__ void grid_partials(const GridRed &g, double (&v)[NS + NM]) {
    constexpr int NV = NS + NM;
    static_assert(NV <= kMaxRedValues, "too many reduced values");
    __shared__ double lds[NV * 16];
    block_reduce<NS, NM>(v, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) g.partials[(size_t)i * kMaxRedBlocks + blockIdx.x] = v[i];
}

// No follow-up work after a reduction.
struct NoTail {
    template <class S> __device__ void operator()(const double *, S *) const {}
};

// One workgroup folds the partial packs of `nblocks` workgroups in a fixed
// order (thread t takes blocks t, t + 256, ... into four accumulators, so four
// loads are in flight), writes g.out and hands the values to
// tail(values, scalars) in thread 0.
// gate: skip everything when *gate == 0 (device-resident loops).
template <int NS, int NM, class Tail, class S>
__global__ void __launch_bounds__(kBlock) grid_fold_kernel(GridRed g, int nblocks, Tail tail, S *scalars,
                                                            const int *gate) {
    if (gate && *gate == 0) return;
    constexpr int NV = NS + NM;
    __shared__ double lds[NV * 16];
    double t[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const double id = i < NS ? 0.0 : -INFINITY;
        const double *P = g.partials + (size_t)i * kMaxRedBlocks;
        double a[4] = {id, id, id, id};
        for (int b0 = threadIdx.x; b0 < nblocks; b0 += 4 * kBlock)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b = b0 + q * kBlock;
                a[q] = combine<NS>(i, a[q], b < nblocks ? P[b] : id);
            }
        t[i] = combine<NS>(i, combine<NS>(i, a[0], a[1]), combine<NS>(i, a[2], a[3]));
    }
    block_reduce<NS, NM>(t, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) g.out[i] = t[i];
        tail(t, scalars);
    }
}

inline int blocks_for(long long n, int per_block = kBlock, int cap = kMaxRedBlocks) {
    long long b = (n + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (int)b;
}

// |x| for the infinity norm; a non-finite entry makes the norm infinite
// (reference src/utils.cu:563-564).
__device__ __forceinline__ double abs_or_inf(double x) { return isfinite(x) ? fabs(x) : INFINITY; }

}  // namespace pdhcg
