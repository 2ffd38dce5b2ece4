// device_common.hpp -- gfx950 device helpers shared by every kernel file.
//
//  * 256-thread blocks = 4 wavefronts of 64 lanes.
//  * Grids are "persistent": G blocks (a multiple of the 8 XCDs) each own
//    a contiguous range of tiles.  The hardware hands block b to XCD b % 8,
//    so the logical block lb = (b % 8) * (G / 8) + b / 8 gives every XCD one
//    contiguous slab of rows: stencil neighbours of a row (the +-nx and
//    +-nx*ny columns) are then read by the same XCD and hit its L2.
//  * Reductions are deterministic: a fixed per-thread order, a fixed
//    butterfly inside the wavefront, a fixed order across waves, one partial
//    per logical block; the consuming kernel sums the partials in
//    logical-block order (strided_sum), in every block that needs them.
#pragma once

#include <hip/hip_runtime.h>

namespace cel {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kXcds = 8;

__device__ __forceinline__ int logical_block()
{
    const int G = gridDim.x;
    const int b = blockIdx.x;
    if (G % kXcds) return b;
    return (b % kXcds) * (G / kXcds) + b / kXcds;
}

// Streaming loads of the matrix: read once per SpMV, keep them out of L2 so
// the gathered vector stays resident.
template <typename T>
__device__ __forceinline__ T ld_stream(const T* p)
{
    return __builtin_nontemporal_load(p);
}

// A 16-byte load; NT: of data that is not wanted in the caches any more.
template <bool NT, typename V>
__device__ __forceinline__ V ld_vec(const void* p)
{
    typedef unsigned int U4 __attribute__((ext_vector_type(4)));
    static_assert(sizeof(V) == 16, "one 16-byte load");
    if constexpr (NT) return __builtin_bit_cast(V, __builtin_nontemporal_load((const U4*)p));
    else return *(const V*)p;
}

// Lane exchanges of the butterfly sums, in registers: halves of the wave and
// of its 32-lane halves through the swap instructions, the rest through
// DPP.  (Through LDS, as __shfl_xor does it, a wave sum took 490 cycles; so
// it takes 190, and every kernel of a solver iteration has two to four of
// them in its chain.)
__device__ __forceinline__ double lanes_f64(unsigned lo, unsigned hi)
{
    return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

// v[l] + v[l ^ 32] and v[l] + v[l ^ 16]
__device__ __forceinline__ double add_xor32(double v)
{
    const auto u = __builtin_bit_cast(unsigned long long, v);
    const auto a = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    return lanes_f64(a[0], b[0]) + lanes_f64(a[1], b[1]);
}
__device__ __forceinline__ double add_xor16(double v)
{
    const auto u = __builtin_bit_cast(unsigned long long, v);
    const auto a = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    return lanes_f64(a[0], b[0]) + lanes_f64(a[1], b[1]);
}
template <int CTRL>
__device__ __forceinline__ double add_dpp(double v)
{
    const auto u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (unsigned)u, CTRL, 0xf, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (unsigned)(u >> 32), CTRL, 0xf, 0xf, false);
    return v + lanes_f64(lo, hi);
}
// v[l] + v[l ^ 8]: rows of 16 lanes rotated by 8
__device__ __forceinline__ double add_xor8(double v) { return add_dpp<0x128>(v); }
// v[l] + v[l ^ 4] of values that repeat with period 8: rows rotated by 4
__device__ __forceinline__ double add_xor4_of8(double v) { return add_dpp<0x124>(v); }
// v[l] + v[l ^ 2] and v[l] + v[l ^ 1]: quad permutations
__device__ __forceinline__ double add_xor2(double v) { return add_dpp<0x4E>(v); }
__device__ __forceinline__ double add_xor1(double v) { return add_dpp<0xB1>(v); }

// Sum of the wave's lanes in every lane: the butterfly over lane distances
// 32, 16, 8, 4, 2, 1.
__device__ __forceinline__ double wave_sum(double v)
{
    return add_xor1(add_xor2(add_xor4_of8(add_xor8(add_xor16(add_xor32(v))))));
}

// Sum over the block in every thread, in block_sum's order.  smem must not be
// written again before the block's next barrier.
__device__ __forceinline__ double block_sum_all(double v, double* smem /* kWaves */)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s = s + smem[w];
    return s;
}

// Sum over the block; valid in thread 0.  Order: butterfly in each wave,
// then waves 0..3 in order.
__device__ __forceinline__ double block_sum(double v, double* smem /* kWaves */)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
        for (int w = 0; w < kWaves; ++w) s = s + smem[w];
    }
    __syncthreads();
    return s;
}

// Two sums at once (same order as block_sum).
__device__ __forceinline__ void block_sum2(double& a, double& b, double* smem /* 2*kWaves */)
{
    a = wave_sum(a);
    b = wave_sum(b);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        smem[wave] = a;
        smem[kWaves + wave] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double sa = 0.0, sb = 0.0;
        for (int w = 0; w < kWaves; ++w) {
            sa = sa + smem[w];
            sb = sb + smem[kWaves + w];
        }
        a = sa;
        b = sb;
    }
    __syncthreads();
}

// The calling thread's part of a fold of G partials: t, t + 256, ...
// in order; block_sum_all of the parts is the fold.  Every block of the
// consuming kernel reads the same partials, so they are plain (cached)
// loads: after the first block on an XCD the rest hit its L2.
__device__ __forceinline__ double strided_sum(const double* __restrict__ partials, int G)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < G; i += kBlock) s = s + partials[i];
    return s;
}

// strided_sum in two parts: the loads (the first four of a thread, none of
// them waited for here) and, later, their sum in the same order.  As loops,
// two folds in a row were two round trips to memory, both ahead of every
// other load of the kernel.  ALL: all four are loaded whatever the count, in
// place of a uniform branch each (32^3 FP64 10.9 / 11.2 us per iteration, but
// mixed 12.8 / 12.6, JAD 61x47x73 15.2 / 14.7).
template <bool ALL>
struct Parts {
    static constexpr int kAhead = 4;
    double a[kAhead];
    const double* p;
    int G;
    __device__ __forceinline__ Parts(const double* partials, int count) : p(partials), G(count)
    {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            a[k] = 0.0;
            const int i = threadIdx.x + k * kBlock;
            if (ALL || k == 0 || G > k * kBlock) a[k] = partials[i < G ? i : 0];
        }
    }
    __device__ __forceinline__ double sum() const
    {
        double s = 0.0;  // (a sum that starts so is never -0: adding +0 keeps it)
#pragma unroll
        for (int k = 0; k < kAhead; ++k) s = s + ((int)threadIdx.x + k * kBlock < G ? a[k] : 0.0);
        for (int i = threadIdx.x + kAhead * kBlock; i < G; i += kBlock) s = s + p[i];
        return s;
    }
};

}  // namespace cel
