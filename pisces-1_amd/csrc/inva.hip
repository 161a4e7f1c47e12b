// inva.hip -- the inverse polarization matrix of PolType 3 on the GPU.
//
// InvA = (alpha^-1 - T)^-1 over the polarizable sites (ComputeInvA,
// src/MolPolAux.cpp:39-136), n = 3 np <= 576.  For a physical set of sites the
// matrix is positive definite, and a blocked Gauss-Jordan elimination needs no
// pivoting: per 16-column block K, with D = A_KK^-1,
//   A_ij -= A_iK D A_Kj,   A_iK <- -A_iK D,   A_Kj <- D A_Kj,   A_KK <- D.
// Its 16 x 16 pivots are the Schur complements of the Cholesky factorisation, so
// a pivot that is not positive shows a matrix that is not positive definite
// (the flag; the caller then takes the host's pivoted elimination).
//
// A step is one launch from one copy of the matrix to another.  It is bound by
// the latency of the chain through D, so every workgroup (64 x 64 elements, one
// 16-row block per wave) inverts D itself, one wave with four elements a lane,
// while the other operands are on their way; the products run on
// v_mfma_f64_16x16x4f64.  A step takes 7 us (5 us of it launch and load
// latency): 0.10 ms for n = 216 and 0.19 ms for n = 405, where the host's
// Cholesky inverse took 5.3 ms and held the GPU idle.
#include "common.hpp"
#include "gmem.hpp"

#include <utility>

namespace pisces {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mma(double a, double b, f64x4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// A = alpha^-1 - T with the Thole-damped dipole tensor T = 3 f5 R R^T / r^5 -
// f3 I / r^3, x = 0.3 r^3 / sqrt(alpha_i alpha_j), f3 = 1 - e^-x, f5 = 1 -
// (1 + x) e^-x between every pair; the identity in the padding.  One thread an
// element.
__global__ void __launch_bounds__(256)
inva_build_kernel(int np, int n3p, const double *__restrict__ rpol, const double *__restrict__ alpha,
                  double *__restrict__ A, int *__restrict__ flag)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e == 0) *flag = 0;
    if (e >= n3p * n3p) return;
    const int r = e / n3p, c = e - r * n3p, i = r / 3, j = c / 3, u = r % 3, w = c % 3;
    double v = 0.0;
    if (i >= np || j >= np) {
        v = r == c ? 1.0 : 0.0;
    } else if (i == j) {
        v = u == w ? 1.0 / alpha[i] : 0.0;
    } else {
        const double d[3] = {rpol[3 * i] - rpol[3 * j], rpol[3 * i + 1] - rpol[3 * j + 1],
                             rpol[3 * i + 2] - rpol[3 * j + 2]};
        const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        const double rr = sqrt(r2), r3 = rr * r2, r5 = r3 * r2;
        const double x = 0.3 * r3 / sqrt(alpha[i] * alpha[j]), ex = exp(-x);
        const double f3 = 1.0 - ex, f5 = 1.0 - (1.0 + x) * ex;
        const double du = u == 0 ? d[0] : u == 1 ? d[1] : d[2], dw = w == 0 ? d[0] : w == 1 ? d[1] : d[2];
        v = -(3.0 * f5 * du * dw / r5 - (u == w ? f3 / r3 : 0.0));
    }
    A[e] = v;
}

// Step K of the elimination, In -> Out (n3p x n3p, n3p a multiple of 16).
__global__ void __launch_bounds__(256)
inva_step_kernel(const double *__restrict__ In_, double *__restrict__ Out_, int n3p, int K,
                 int *__restrict__ flag)
{
    __shared__ double D[16][17];
    __shared__ double Ws[4][16][17];
    const gptr<const double> In = glb(In_);
    const gptr<double> Out = glb(Out_);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4, nb = n3p / 16;
    const int rb = 4 * blockIdx.y + wave, cb0 = 4 * blockIdx.x;
    const bool row_in = rb < nb;
    // the wave's operands: its 16 rows of column block K (A form), row block K
    // of its columns (B form), and its tiles
    double aik[4], bkj[4][4];
    f64x4 acc[4];
    if (row_in) {
#pragma unroll
        for (int s = 0; s < 4; ++s) aik[s] = In[(16 * rb + l16) * n3p + 16 * K + 4 * s + lq];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * (cb0 + v < nb ? cb0 + v : 0) + l16;
#pragma unroll
            for (int s = 0; s < 4; ++s) bkj[v][s] = In[(16 * K + 4 * s + lq) * n3p + c];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[v][r] = rb == K ? 0.0 : In[(16 * rb + lq + 4 * r) * n3p + c];
        }
    }
    if (wave == 0) {
        // lane: row lane / 4, columns 4 (lane % 4) ..
        const int i = lane >> 2, j0 = 4 * (lane & 3);
        double x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = In[(16 * K + i) * n3p + 16 * K + j0 + c];
        bool bad = false;
#pragma unroll
        for (int p = 0; p < 16; ++p) {
            const double piv = __shfl(x[p & 3], 4 * p + (p >> 2), 64);
            const double f = __shfl(x[p & 3], (lane & ~3) + (p >> 2), 64);
            double row[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) row[c] = __shfl(x[c], 4 * p + (lane & 3), 64);
            bad = bad || !(piv > 0.0);
            const double inv = rcp64(piv);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bool col = j0 + c == p;
                if (i == p) x[c] = col ? inv : x[c] * inv;
                else x[c] = col ? -f * inv : x[c] - f * (row[c] * inv);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) D[i][j0 + c] = x[c];
        if (bad && lane == 0 && blockIdx.x == 0 && blockIdx.y == 0) *flag = 1;
    }
    __syncthreads();
    if (!row_in) return;
    f64x4 w = {0.0, 0.0, 0.0, 0.0};
    if (rb != K) {
#pragma unroll
        for (int s = 0; s < 4; ++s) w = mma(aik[s], D[4 * s + lq][l16], w);  // A_iK D
#pragma unroll
        for (int r = 0; r < 4; ++r) Ws[wave][lq + 4 * r][l16] = -w[r];
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) Ws[wave][lq + 4 * r][l16] = D[lq + 4 * r][l16];
    }
    wave_lds_sync();
    double a[4];  // -A_iK D, or D in row block K, in A form
#pragma unroll
    for (int s = 0; s < 4; ++s) a[s] = Ws[wave][l16][4 * s + lq];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int cb = cb0 + v;
        if (cb >= nb) break;
        if (cb == K) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[v][r] = rb == K ? D[lq + 4 * r][l16] : -w[r];
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[v] = mma(a[s], bkj[v][s], acc[v]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) Out[(16 * rb + lq + 4 * r) * n3p + 16 * cb + l16] = acc[v][r];
    }
}

// Both triangles from the lower one, zero outside the leading n x n; flags a
// value that is not finite.
__global__ void __launch_bounds__(256)
inva_finish_kernel(const double *__restrict__ A, int n, int n3p, double *__restrict__ inva,
                   int *__restrict__ flag)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n3p * n3p) return;
    const int r = e / n3p, c = e - r * n3p;
    double v = 0.0;
    if (r < n && c < n) v = r >= c ? A[e] : A[c * n3p + r];
    if (!(fabs(v) < __builtin_huge_val())) *flag = 1;
    inva[e] = v;
}

}  // namespace

void pol3_inva_launch(int np, const double *d_rpol, const double *d_alpha, int n3p, double *d_tmp,
                      double *d_inva, int *d_flag, hipStream_t s)
{
    PC_REQUIRE(np > 0 && n3p == pol3_padded(np) && n3p <= kPol3MaxN, PISCES_ERR_UNSUPPORTED,
               "too many polarizable sites");
    const size_t nn = (size_t)n3p * n3p;
    const unsigned blocks = (unsigned)((nn + 255) / 256), t = (unsigned)((n3p + 63) / 64);
    double *in = d_tmp, *out = d_tmp + nn;
    hipLaunchKernelGGL(inva_build_kernel, dim3(blocks), dim3(256), 0, s, np, n3p, d_rpol, d_alpha, in,
                       d_flag);
    for (int K = 0; K < n3p / 16; ++K) {
        hipLaunchKernelGGL(inva_step_kernel, dim3(t, t), dim3(256), 0, s, in, out, n3p, K, d_flag);
        std::swap(in, out);
    }
    hipLaunchKernelGGL(inva_finish_kernel, dim3(blocks), dim3(256), 0, s, in, 3 * np, n3p, d_inva, d_flag);
    PC_HIP(hipGetLastError());
}

}  // namespace pisces
