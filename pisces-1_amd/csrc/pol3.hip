// pol3.hip -- the self-consistent polarization potential (PolType 3) on the grid.
//
// Potential::SelfConsistentPolarizability (src/Potential.cpp:1495-1592) at a
// grid point r: E_i = g(R_i) R_i + Epc_i at the polarizable sites i (R_i =
// r - site i, g the damped R^-3), mu = InvA E, Vpol = -E.mu / 2 -
// VpolWaterWater.  Over a tile of grid points that is the product E InvA (points
// x 3np times 3np x 3np) followed by a row-wise dot with E: FP64 matrix-core
// work of 2 (3np)^2 flops per point.  InvA is symmetric, so only its upper block
// triangle is multiplied: (3np)^2 (1 + 16 / 3np) flops per point.  A workgroup
// takes 16 RB points (RB = 2 by default): it builds their E rows in LDS (odd
// pitch: the 16 rows that one matrix-core operand reads fall on distinct banks),
// then its waves split the list of 16 x 16 InvA tiles evenly, stream them from
// L2 (InvA is shared by all workgroups: at most 2.6 MB) one tile ahead as the B
// operand of v_mfma_f64_16x16x4 against the row blocks of E, and fold each column
// block's sum into the per-point dot.  us at 216 / 405 dimensions, before (16
// points, whole column blocks per wave, 64-bit divisions for every E value) ->
// now: 423 / 4360 -> 341 / 3311, which is 0.57 / 0.64 of the 72.7 TFLOP/s that a
// large FP64 matrix product reaches; the E rows and the ends of a workgroup are
// the rest.
#include "common.hpp"
#include "gmem.hpp"

#include <cstdlib>
#include <mutex>

namespace pisces {

namespace {

constexpr int kLdsMax = 160 * 1024 - (16 + 3) * 64 * (int)sizeof(double);  // E rows, red (16 waves), pt

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ inline double reff3(double r, double r0)
{
    // effective-distance damping, src/Potential.cpp:1191-1196
    if (r < r0) {
        const double t = r / r0;
        return r0 * (0.5 + t * t * t * (1.0 - 0.5 * t));
    }
    return r;
}

// RB 16-point row blocks per workgroup (kP3Pts = 16 RB grid points), NT threads
template <int RB, int NT>
__global__ void __launch_bounds__(NT)
pol3_grid_kernel(Pol3Dev D, int nx, int ny, int nz, const double *__restrict__ gx,
                 const double *__restrict__ gy, const double *__restrict__ gz,
                 double *__restrict__ v)
{
    constexpr int kP3Pts = 16 * RB, kP3Threads = NT, NW = NT / 64;
    extern __shared__ double Es[];  // kP3Pts rows of n3p (+1) values
    __shared__ double red[kP3Threads / 64][kP3Pts];
    __shared__ double pt[kP3Pts][3];  // the points' coordinates
    const int n3p = D.n3p, ldE = n3p + 1, np = D.np, n3 = 3 * np;
    const long long ng = (long long)nx * ny * nz;
    const long long g0 = (long long)blockIdx.x * kP3Pts;
    const gptr<const double> rp = glb(D.rpol), ep = glb(D.epc);

    // E rows: the electron's field at the sites (src/Potential.cpp:1531-1562,
    // DampType 1: R^-3 (1 - exp(-p R^3)); 2: Reff^-3 inside the damping radius)
    // plus the permanent-charge field; rows past the grid repeat its last point
    if (threadIdx.x < kP3Pts) {
        const unsigned g = (unsigned)(g0 + threadIdx.x < ng ? g0 + threadIdx.x : ng - 1);
        const unsigned iy = g / (unsigned)nx, iz = iy / (unsigned)ny;
        pt[threadIdx.x][0] = gx[g - iy * nx];
        pt[threadIdx.x][1] = gy[iy - iz * ny];
        pt[threadIdx.x][2] = gz[iz];
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < kP3Pts * np; idx += kP3Threads) {
        const int p = idx % kP3Pts, i = idx / kP3Pts;
        const double rx = pt[p][0] - rp[3 * i], ry = pt[p][1] - rp[3 * i + 1], rz = pt[p][2] - rp[3 * i + 2];
        const double R2 = rx * rx + ry * ry + rz * rz;
        double gij = 0.0;  // R = 0: the field's limit, 0
        if (R2 > 0.0) {
            const double ri = rsq64(R2), R = R2 * ri;
            if (D.damp_type == 1) {
                gij = ri * ri * ri * (1.0 - exp(-D.pdamp * R * R2));
            } else if (R < D.pdamp) {
                const double re = reff3(R, D.pdamp);
                gij = rcp64(re * re * re);
            } else {
                gij = ri * ri * ri;
            }
        }
        double *row = Es + p * ldE + 3 * i;
        row[0] = gij * rx + ep[3 * i];
        row[1] = gij * ry + ep[3 * i + 1];
        row[2] = gij * rz + ep[3 * i + 2];
    }
    for (int idx = threadIdx.x; idx < kP3Pts * (n3p - n3); idx += kP3Threads)
        Es[(idx % kP3Pts) * ldE + n3 + idx / kP3Pts] = 0.0;
    __syncthreads();

    // E^T InvA E over the upper block triangle of the symmetric InvA: 16 x 16
    // tiles above the diagonal count twice, those on it once.  The tiles, column
    // by column, are one list that the waves split evenly; a wave folds its sum
    // over the rows k of a column block into the per-point dot when it leaves
    // the column.  The next tile's InvA values are requested before the current
    // ones are used.
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const gptr<const double> A = glb(D.inva) + (lq * n3p + l16);
    double sr[RB][4];
    f64x4 o[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        o[b] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int r = 0; r < 4; ++r) sr[b][r] = 0.0;
    }
    const double *ea = Es + l16 * ldE + lq;  // row block b: + 16 b ldE
    const int ncb = n3p / 16, ntile = ncb * (ncb + 1) / 2;
    const int t0 = ntile * wave / NW, t1 = ntile * (wave + 1) / NW;
    // tile t0: column block cb, row block kb <= cb
    int cb = 0, kb = t0;
    while (kb > cb) {
        kb -= cb + 1;
        ++cb;
    }
    double nv[4];
    if (t0 < t1)
#pragma unroll
        for (int q = 0; q < 4; ++q) nv[q] = A[(16 * kb + 4 * q) * n3p + 16 * cb];
    auto fold = [&](double w) {
        const int c = 16 * cb + l16;
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sr[b][r] += (w * o[b][r]) * Es[(16 * b + lq + 4 * r) * ldE + c];
                o[b][r] = 0.0;
            }
    };
    for (int t = t0; t < t1; ++t) {
        const bool diag = kb == cb;
        const int nk = diag ? 0 : kb + 1, nc = diag ? cb + 1 : cb;  // the next tile
        double bv[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[q] = nv[q];
        if (t + 1 < t1)
#pragma unroll
            for (int q = 0; q < 4; ++q) nv[q] = A[(16 * nk + 4 * q) * n3p + 16 * nc];
        if (diag) fold(2.0);  // the tiles above the diagonal so far
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int b = 0; b < RB; ++b)
                o[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(ea[16 * b * ldE + 16 * kb + 4 * q], bv[q], o[b], 0, 0, 0);
        if (diag) fold(1.0);
        if (t + 1 == t1 && !diag) fold(2.0);
        kb = nk;
        cb = nc;
    }
    // sum over the 16 columns a lane group holds, then over the waves
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) sr[b][r] = row_sum(sr[b][r]);
    if (l16 == 0)
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][16 * b + lq + 4 * r] = sr[b][r];
    __syncthreads();
    if (threadIdx.x < kP3Pts) {
        const long long g = g0 + threadIdx.x;
        if (g < ng) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < kP3Threads / 64; ++w) s += red[w][threadIdx.x];
            v[g] += -0.5 * s - D.vpolww;
        }
    }
}

}  // namespace

void pol3_grid_launch(const Pol3Dev &D, int nx, int ny, int nz, const double *d_x,
                      const double *d_y, const double *d_z, double *d_v, hipStream_t s)
{
    PC_REQUIRE(D.np > 0 && D.n3p == pol3_padded(D.np) && D.n3p <= kPol3MaxN,
               PISCES_ERR_UNSUPPORTED, "too many polarizable sites");
    PC_REQUIRE(D.damp_type == 1 || D.damp_type == 2, PISCES_ERR_ARG, "damping type");
    static std::once_flag once;
    std::call_once(once, [] {
        const void *ks[] = {reinterpret_cast<const void *>(pol3_grid_kernel<1, 256>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<2, 256>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<4, 256>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<1, 512>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<2, 512>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<4, 512>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<1, 1024>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<2, 1024>),
                            reinterpret_cast<const void *>(pol3_grid_kernel<4, 1024>)};
        for (const void *k : ks)
            PC_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax));
    });
    // RB 16-point row blocks per workgroup (PISCES_POL3_RB = 1, 2 or 4): each
    // InvA fragment from the L2 feeds RB products, the E rows in LDS bound the
    // workgroups per CU.  us at 216 (64^3) / 405 dimensions (96^3), RB 1, 2, 4
    // with the threads below: 359 / 3377, 341 / 3311, 381 / 3325.
    const char *rb_e = std::getenv("PISCES_POL3_RB");  // read per build: not a hot path
    const int rb_env = rb_e ? std::atoi(rb_e) : 0;
    // threads per workgroup (PISCES_POL3_NT = 256, 512 or 1024): 512 as long as
    // the LDS of two workgroups with 32-point tiles fits a CU (19 column blocks),
    // 1024 beyond.  us at 64^3, 512 / 1024 threads, by column blocks (waters): 14
    // (24) 332 / 399, 18 (32) 506 / 572, 19 (33) 556 / 638, 20 (34) 750 / 690, 23 (40)
    // 937 / 876, 26 (45) 1157 / 1045, 36 (64) 2075 / 1851; the same line at 48^3.
    const char *nt_e = std::getenv("PISCES_POL3_NT");
    const int nt_v = nt_e ? std::atoi(nt_e) : (D.n3p / 16 >= 20 ? 1024 : 512);
    const int nt = (nt_v == 256 || nt_v == 1024) ? nt_v : 512;
    const size_t row = (size_t)(D.n3p + 1) * sizeof(double);
    int rb = (rb_env == 1 || rb_env == 2 || rb_env == 4) ? rb_env : 2;
    while (rb > 1 && 16 * rb * row > (size_t)kLdsMax) rb /= 2;
    const long long ng = (long long)nx * ny * nz;
    const int pts = 16 * rb;
    const unsigned blocks = (unsigned)((ng + pts - 1) / pts);
    const size_t lds = (size_t)pts * row;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(nt), lds, s, D, nx, ny, nz, d_x, d_y, d_z, d_v);
    };
    if (nt == 1024) go(rb == 1 ? pol3_grid_kernel<1, 1024> : rb == 2 ? pol3_grid_kernel<2, 1024> : pol3_grid_kernel<4, 1024>);
    else if (nt == 512) go(rb == 1 ? pol3_grid_kernel<1, 512> : rb == 2 ? pol3_grid_kernel<2, 512> : pol3_grid_kernel<4, 512>);
    else go(rb == 1 ? pol3_grid_kernel<1, 256> : rb == 2 ? pol3_grid_kernel<2, 256> : pol3_grid_kernel<4, 256>);
    PC_HIP(hipGetLastError());
}

}  // namespace pisces
