// plane.hpp -- what the matrix-core plane kernels share (plane.hip: split-BF16
// forms, plane_f.hip: FP64 and FP32 forms): operand types, plane geometry, grid
// numbering and launch helpers.  Device helpers are per translation unit.
#pragma once

#include "common.hpp"
#include "fdm.hpp"
#include "gmem.hpp"

namespace pisces {

// FP64 and FP32 forms (plane_f.hip).  max_planes_a, _b: the largest number of
// planes of a job in pass A and B; max_n: the largest axis of any job or task.
// `one`, where not null, replaces the d_jobs / d_tasks in memory.
void hx_f_launch(const HxJob *d_jobs, const HxJob *one, int njobs, int max_planes_a, int max_planes_b, int max_n,
                 int precision, hipStream_t s);
void fdm_f64_launch(const FdmTask *d_tasks, const FdmOne *one, int ntasks, int max_n, hipStream_t s);

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f64x4 mma(double a, double b, f64x4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename T> struct Acc;
template <> struct Acc<double> {
    typedef f64x4 type;
    __device__ static inline int row(int lq, int r) { return lq + 4 * r; }
};
template <> struct Acc<float> {
    typedef f32x4 type;
    __device__ static inline int row(int lq, int r) { return 4 * lq + r; }
};

// Plane geometry.  kind 0: plane (i,j) at fixed k (rows c = j); kind 1: plane
// (i,k) at fixed j (rows c = k).
struct Geo {
    int ni, nc, npi, npc;
    long long cs;     // global stride between rows
    long long vbase;  // offset of (0, 0) within one vector
    long long base;   // offset of (0, 0) including the vector offset
    int pl;           // index of the plane along its normal axis
};

__device__ __forceinline__ bool geo_of(int kind, int nx, int ny, int nz, int nvec, long long ld,
                                       int npi, int npc, int p, Geo &g)
{
    const int nplanes = kind == 0 ? nz : ny;
    if (p >= nplanes * nvec) return false;
    const int v = p / nplanes, pl = p - v * nplanes;
    g.ni = nx;
    g.npi = npi;
    g.npc = npc;
    g.pl = pl;
    if (kind == 0) {
        g.nc = ny;
        g.cs = nx;
        g.vbase = (long long)nx * ny * pl;
    } else {
        g.nc = nz;
        g.cs = (long long)nx * ny;
        g.vbase = (long long)nx * pl;
    }
    g.base = (long long)v * ld + g.vbase;
    return true;
}

// The middle pass of H*X (pass B) and of the preconditioner (pass 1) reads
// what the pass before wrote: it walks its grid in reverse (workgroups are
// dispatched in order of their linear index), starting on the data the
// previous pass left last in the L2 and the memory-side cache.
__device__ __forceinline__ int plane_x(bool rev) { return rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x; }
__device__ __forceinline__ int plane_y(bool rev) { return rev ? gridDim.y - 1 - blockIdx.y : blockIdx.y; }

// task of vector blockIdx.y (reversed as plane_y) of a grid passed by value;
// elements of es_src, es_dst bytes
__device__ __forceinline__ FdmTask task_of(const FdmOne &one, int v, int es_src, int es_dst)
{
    FdmTask t = one.t;
    t.src = static_cast<const char *>(t.src) + one.ngp * v * es_src;
    t.dst = static_cast<char *>(t.dst) + one.ngp * v * es_dst;
    t.work += one.ngp * v;
    return t;
}

// Raises a kernel's dynamic LDS limit to `bytes` (the 160 KB of a CU less the
// kernel's static LDS); a failure is reported, not left behind as the thread's
// last HIP error.
template <typename K>
void allow_lds(K kernel, size_t bytes = 160 * 1024)
{
    PC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

}  // namespace

}  // namespace pisces
