// gmem.hpp -- address-space pointers and FP64 reciprocals for device code.
//
// Pointers that kernels read out of task descriptors are generic to the
// compiler, which then emits flat memory instructions: they count against both
// the vector-memory and the LDS counters, so LDS waits also wait for HBM loads
// and loads guarded by conditions become branches.  Casting such pointers to
// the global address space gives global_load / global_store instead.
#pragma once

#include <hip/hip_runtime.h>

namespace pisces {

template <typename T> using gptr = __attribute__((address_space(1))) T *;

template <typename T> __device__ __forceinline__ gptr<T> glb(T *p) { return (gptr<T>)p; }

// Constant address space: for data that no thread writes while the kernel
// runs (coefficients produced by earlier launches).  Wave-uniform loads
// through it become scalar loads; vector stores elsewhere in the kernel
// (possibly of the same type) no longer force them onto the vector path.
template <typename T> using cptr = __attribute__((address_space(4))) const T *;

template <typename T> __device__ __forceinline__ cptr<T> cst(const T *p) { return (cptr<T>)p; }

// Loads of block columns that one workgroup of a launch streams through once
// carry the nontemporal hint (the nt bit): on MI355X a plain read stream of
// 1 GiB measured 7.1 TB/s with it against 6.3 TB/s with the default policy
// (pisces_stream_probe).  Columns that several workgroups of the same launch
// read again from the L2 keep the default policy.
template <typename T> __device__ __forceinline__ T ldnt(gptr<const T> p)
{
    return __builtin_nontemporal_load(p);
}
template <typename T> __device__ __forceinline__ T ldnt(const T *p)
{
    return __builtin_nontemporal_load(p);
}

// Stores of outputs that no later work of the same launch reads again, with
// the nontemporal hint.
template <typename T> __device__ __forceinline__ void stnt(gptr<T> p, T v)
{
    __builtin_nontemporal_store(v, p);
}

// 1/x and 1/sqrt(x) in FP64 to about one ulp.  The reciprocal: the hardware
// estimate refined by two Newton-Raphson steps, r <- r + r (1 - x r), each
// squaring the relative error.  The root: one cubic step, y <- y + y e (1/2 + 3 e / 8)
// with e = 1 - x y^2, which leaves 5 e^3 / 16 of an estimate good to single
// precision (below 2^-65), the rounding of x y in e and that of the last sum, in
// five operations.  Against 80-bit arithmetic, 4 M arguments in 2^-8 .. 2^14: at
// most 0.99 ulp, 0.33 rms; two quadratic steps in eight operations: 1.64, 0.47.
__device__ __forceinline__ double rcp64(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    r = fma(r, fma(-x, r, 1.0), r);
    return r;
}
__device__ __forceinline__ double rsq64(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// x plus x of the lane that a DPP control names, and sums over groups of lanes
// by them (the LDS stays out of it): quad permutes 1,0,3,2 (0xB1) and 2,3,0,1
// (0x4E), then, on equal quads and equal groups of 8, the half-row (0x141) and
// row (0x140) mirrors.
template <int CTRL> __device__ __forceinline__ double dpp_add(double x)
{
    const long long v = __builtin_bit_cast(long long, x);
    const int lo = __builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), CTRL, 0xF, 0xF, false);
    return x + __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// the sum of the 16 lanes of a row, in all of them
__device__ __forceinline__ double row_sum(double x)
{
    return dpp_add<0x140>(dpp_add<0x141>(dpp_add<0x4E>(dpp_add<0xB1>(x))));
}

// Between a wave's writes to LDS and its lanes' reads of each other's: the
// hardware runs a wave's LDS operations in order, and this keeps the compiler
// from moving them across (no instruction, no wait).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lane l's value of x, uniform over the wave
__device__ __forceinline__ double lane_value(double x, int l)
{
    const long long v = __builtin_bit_cast(long long, x);
    const int lo = __builtin_amdgcn_readlane((int)v, l);
    const int hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// the sum of the 64 lanes of a wave, in all of them
__device__ __forceinline__ double lanes_sum(double x)
{
    const double r = row_sum(x);
    return (lane_value(r, 0) + lane_value(r, 16)) + (lane_value(r, 32) + lane_value(r, 48));
}

}  // namespace pisces
