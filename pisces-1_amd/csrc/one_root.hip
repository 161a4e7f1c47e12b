// one_root.hip -- kernels of the one-root FP64 Davidson solve (solver_fp64.cpp).
//
// An iteration for one root works on a dozen columns of a few hundred kilobytes:
// launches, the host's turn and the gaps between them cost more than the data.
// The iteration is therefore four kernels around H*X with one wait for the host,
// each fusing a pass over the subspace with the dot products that the next one
// needs (B, Z: the m columns of the subspace and of H B; y, theta: the Ritz pair):
//   ritz1:  u = B y, z = Z y, r = z - theta u, c = r / (theta - diag H); ||r||^2,
//           ||u||^2, h = B^T c
//   orth1:  c <- c - B h; h2 = B^T c, ||c||^2
//   orth2:  b = (c - B h2) / sqrt(||c||^2 - ||h2||^2), the new column of B
//   dots1:  (after z = H b) Z^T b, the new column of the projected matrix, ||b||^2
//   finish1: the sums that the host reads, into its memory
// The dot products leave one row of partial sums per workgroup, which every
// workgroup of the next kernel adds for itself in the same order.
#include "blockops.hpp"
#include "gmem.hpp"

namespace pisces {

namespace {

constexpr int kT = 256;
constexpr int kLd = kOneLd;  // doubles per row of partial sums
constexpr int kRows = 256;   // rows of partial sums that a kernel still adds itself

// LDS of a workgroup's dot products: 16 partial sums (4 waves x 4 rows of lanes)
// of every value.
struct Dots {
    double v[kLd][17];
};

// value `i` of this thread: into the workgroup's sums
__device__ __forceinline__ void dot_put(Dots &d, int i, double x)
{
    x = row_sum(x);
    if ((threadIdx.x & 15) == 0) d.v[i][threadIdx.x >> 4] = x;
}
// the workgroup's row of n partial sums
__device__ __forceinline__ void dot_store(const Dots &d, int n, double *part)
{
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kT) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) s += d.v[i][q];
        part[(size_t)blockIdx.x * kLd + i] = s;
    }
}
// sums of values 0 .. n - 1 over the rows of part, in h (n <= 64)
__device__ __forceinline__ void sum_rows(const double *__restrict__ part, int rows, int n, double (*tmp)[64],
                                         double *h)
{
    const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (i < n) {
        int r = q;
        for (; r + 12 < rows; r += 16)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += part[(size_t)(r + 4 * u) * kLd + i];
        for (; r < rows; r += 4) s[0] += part[(size_t)r * kLd + i];
    }
    tmp[q][i] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (q == 0) h[i] = (tmp[0][i] + tmp[1][i]) + (tmp[2][i] + tmp[3][i]);
    __syncthreads();
}

struct OneCoef {
    double y[kOneMaxM], theta;
};
static_assert(kOneMaxM == 64, "sum_rows: a lane of a wave per sum");

// The RPT rows of a thread; rows past N read row 0 and count as zeros.
template <int RPT> struct Rows {
    unsigned g[RPT];
    bool ok[RPT];
    __device__ __forceinline__ explicit Rows(long long N)
    {
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            const long long r = (long long)blockIdx.x * (kT * RPT) + t * kT + threadIdx.x;
            ok[t] = r < N;
            g[t] = ok[t] ? (unsigned)r : 0u;
        }
    }
};

// sum over the rows of A_a x for every column a < m, into values i0 + a
template <int RPT>
__device__ __forceinline__ void dots(Dots &d, int i0, const double *A, long long N, int m, const Rows<RPT> &R,
                                     const double (&x)[RPT])
{
    const gptr<const double> a0 = glb(A);
#pragma unroll 4
    for (int a = 0; a < m; ++a) {
        double p = 0.0;
#pragma unroll
        for (int t = 0; t < RPT; ++t) p += a0[a * N + R.g[t]] * x[t];
        dot_put(d, i0 + a, p);
    }
}

template <int RPT, bool STORE>
__global__ void __launch_bounds__(kT)
ritz1_kernel(const double *__restrict__ B, const double *__restrict__ Z, const double *__restrict__ D,
             long long N, int m, OneCoef co, double *__restrict__ C, double *__restrict__ U,
             double *__restrict__ ZV, double *__restrict__ part)
{
    __shared__ Dots d;
    const Rows<RPT> R(N);
    double u[RPT], z[RPT], c[RPT];
#pragma unroll
    for (int t = 0; t < RPT; ++t) u[t] = z[t] = 0.0;
    const gptr<const double> gb = glb(B), gz = glb(Z), gd = glb(D);
#pragma unroll 4
    for (int a = 0; a < m; ++a)
#pragma unroll
        for (int t = 0; t < RPT; ++t) {
            u[t] += gb[a * N + R.g[t]] * co.y[a];
            z[t] += gz[a * N + R.g[t]] * co.y[a];
        }
    double rr = 0.0, uu = 0.0;
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
        const double r = z[t] - co.theta * u[t];
        double dv = co.theta - gd[R.g[t]];  // src/Davidson.cpp:557-566
        if (fabs(dv) < 1e-12) dv = 1e-12;
        c[t] = R.ok[t] ? r / dv : 0.0;
        if (R.ok[t]) {
            rr += r * r;
            uu += u[t] * u[t];
            C[R.g[t]] = c[t];
            if (STORE) {
                U[R.g[t]] = u[t];
                ZV[R.g[t]] = z[t];
            }
        }
    }
    dots<RPT>(d, 0, B, N, m, R, c);
    dot_put(d, m, rr);
    dot_put(d, m + 1, uu);
    dot_store(d, m + 2, part);
}

// c <- c - B h with h the first m sums of pin's rows; dots B^T c (m) and ||c||^2
template <int RPT>
__global__ void __launch_bounds__(kT)
orth1_kernel(const double *__restrict__ B, long long N, int m, const double *__restrict__ pin, int rows,
             double *__restrict__ C, double *__restrict__ part)
{
    __shared__ Dots d;
    __shared__ double tmp[4][64], h[64];
    const Rows<RPT> R(N);
    sum_rows(pin, rows, m, tmp, h);
    const gptr<const double> gb = glb(B);
    double c[RPT], cc = 0.0;
#pragma unroll
    for (int t = 0; t < RPT; ++t) c[t] = C[R.g[t]];
#pragma unroll 4
    for (int a = 0; a < m; ++a)
#pragma unroll
        for (int t = 0; t < RPT; ++t) c[t] -= gb[a * N + R.g[t]] * h[a];
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
        if (R.ok[t]) C[R.g[t]] = c[t];
        else c[t] = 0.0;
        cc += c[t] * c[t];
    }
    dots<RPT>(d, 0, B, N, m, R, c);
    dot_put(d, m, cc);
    dot_store(d, m + 1, part);
}

// b = (c - B h2) / sqrt(||c||^2 - ||h2||^2); zero where that is not positive (the
// correction lies in the subspace)
template <int RPT>
__global__ void __launch_bounds__(kT)
orth2_kernel(const double *__restrict__ B, long long N, int m, const double *__restrict__ pin, int rows,
             const double *__restrict__ C, double *__restrict__ b)
{
    __shared__ double tmp[4][64], h[64];
    const Rows<RPT> R(N);
    sum_rows(pin, rows, m + 1, tmp, h);
    const gptr<const double> gb = glb(B);
    double c[RPT], nn = h[m];
#pragma unroll
    for (int t = 0; t < RPT; ++t) c[t] = C[R.g[t]];
#pragma unroll 4
    for (int a = 0; a < m; ++a) {
        nn -= h[a] * h[a];
#pragma unroll
        for (int t = 0; t < RPT; ++t) c[t] -= gb[a * N + R.g[t]] * h[a];
    }
    const double s = nn > 0.0 ? 1.0 / sqrt(nn) : 0.0;
#pragma unroll
    for (int t = 0; t < RPT; ++t)
        if (R.ok[t]) b[R.g[t]] = c[t] * s;
}

// dots A^T x (m) and ||x||^2
template <int RPT>
__global__ void __launch_bounds__(kT)
dots1_kernel(const double *__restrict__ A, long long N, int m, const double *__restrict__ x,
             double *__restrict__ part)
{
    __shared__ Dots d;
    const Rows<RPT> R(N);
    double v[RPT], xx = 0.0;
#pragma unroll
    for (int t = 0; t < RPT; ++t) {
        v[t] = R.ok[t] ? x[R.g[t]] : 0.0;
        xx += v[t] * v[t];
    }
    dots<RPT>(d, 0, A, N, m, R, v);
    dot_put(d, m, xx);
    dot_store(d, m + 1, part);
}

// the sums of values i0 .. i0 + n - 1 over the rows of part: a workgroup per value
__global__ void __launch_bounds__(64)
finish1_kernel(const double *__restrict__ part, int rows, int i0, const double *__restrict__ part2, int j0,
               int n2, double *__restrict__ out)
{
    // workgroups 0 .. n2 - 1: values j0 .. of part2; then those of part
    const bool second = (int)blockIdx.x < n2;
    const double *p = second ? part2 + j0 + blockIdx.x : part + i0 + (blockIdx.x - n2);
    double s = 0.0;
    for (int r = threadIdx.x; r < rows; r += 64) s += p[(size_t)r * kLd];
    s = row_sum(s);
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// x <- f x, y <- g y
__global__ void __launch_bounds__(kT)
scale1_kernel(const double *x, double f, double *xo, const double *y,
              double g, double *yo, long long N)
{
    const long long i = (long long)blockIdx.x * kT + threadIdx.x;
    if (i >= N) return;
    xo[i] = x[i] * f;
    yo[i] = y[i] * g;
}

}  // namespace

// One row per thread up to 256 workgroups (64 K points), four beyond.
static int one_rpt(long long N) { return N <= (long long)kT * kRows ? 1 : 4; }
int one_rows(long long N) { return (int)((N + kT * one_rpt(N) - 1) / (kT * one_rpt(N))); }

// Rows of partial sums that the next kernel adds: with many workgroups a
// reduction to one row comes first (into row `rows` of part).
static const double *one_reduce(double *part, int &rows, int n, hipStream_t s)
{
    if (rows <= kRows) return part;
    double *out = part + (size_t)rows * kLd;
    hipLaunchKernelGGL(finish1_kernel, dim3(n), dim3(64), 0, s, part, rows, 0, nullptr, 0, 0, out);
    rows = 1;
    return out;
}

void one_ritz(const double *B, const double *Z, const double *D, long long N, int m, const double *y,
              double theta, double *C, double *U, double *ZV, double *part, hipStream_t s)
{
    PC_REQUIRE(m >= 1 && m <= kOneMaxM, PISCES_ERR_ARG, "one-root subspace size");
    OneCoef co;
    for (int a = 0; a < kOneMaxM; ++a) co.y[a] = a < m ? y[a] : 0.0;
    co.theta = theta;
    const dim3 g(one_rows(N)), t(kT);
    if (one_rpt(N) == 1) {
        if (U) hipLaunchKernelGGL((ritz1_kernel<1, true>), g, t, 0, s, B, Z, D, N, m, co, C, U, ZV, part);
        else hipLaunchKernelGGL((ritz1_kernel<1, false>), g, t, 0, s, B, Z, D, N, m, co, C, U, ZV, part);
    } else {
        if (U) hipLaunchKernelGGL((ritz1_kernel<4, true>), g, t, 0, s, B, Z, D, N, m, co, C, U, ZV, part);
        else hipLaunchKernelGGL((ritz1_kernel<4, false>), g, t, 0, s, B, Z, D, N, m, co, C, U, ZV, part);
    }
    PC_HIP(hipGetLastError());
}

void one_orth(const double *B, long long N, int m, double *C, double *b, double *part_h, double *part_n,
              hipStream_t s)
{
    PC_REQUIRE(m >= 1 && m < kOneMaxM, PISCES_ERR_ARG, "one-root subspace size");
    const dim3 g(one_rows(N)), t(kT);
    int r1 = one_rows(N), r2 = one_rows(N);
    const double *h = one_reduce(part_h, r1, m, s);
    if (one_rpt(N) == 1) hipLaunchKernelGGL((orth1_kernel<1>), g, t, 0, s, B, N, m, h, r1, C, part_n);
    else hipLaunchKernelGGL((orth1_kernel<4>), g, t, 0, s, B, N, m, h, r1, C, part_n);
    const double *n = one_reduce(part_n, r2, m + 1, s);
    if (one_rpt(N) == 1) hipLaunchKernelGGL((orth2_kernel<1>), g, t, 0, s, B, N, m, n, r2, C, b);
    else hipLaunchKernelGGL((orth2_kernel<4>), g, t, 0, s, B, N, m, n, r2, C, b);
    PC_HIP(hipGetLastError());
}

void one_dots(const double *A, long long N, int m, const double *x, double *part, hipStream_t s)
{
    PC_REQUIRE(m >= 1 && m <= kOneMaxM, PISCES_ERR_ARG, "one-root subspace size");
    const dim3 g(one_rows(N)), t(kT);
    if (one_rpt(N) == 1) hipLaunchKernelGGL((dots1_kernel<1>), g, t, 0, s, A, N, m, x, part);
    else hipLaunchKernelGGL((dots1_kernel<4>), g, t, 0, s, A, N, m, x, part);
    PC_HIP(hipGetLastError());
}

void one_finish(const double *part, long long N, int i0, int n, const double *part2, int j0, int n2,
                double *out, hipStream_t s)
{
    hipLaunchKernelGGL(finish1_kernel, dim3(n + n2), dim3(64), 0, s, part, one_rows(N), i0, part2, j0, n2, out);
    PC_HIP(hipGetLastError());
}

void one_scale(const double *x, double f, double *xo, const double *y, double g, double *yo, long long N,
               hipStream_t s)
{
    hipLaunchKernelGGL(scale1_kernel, dim3((unsigned)((N + kT - 1) / kT)), dim3(kT), 0, s, x, f, xo, y, g, yo, N);
    PC_HIP(hipGetLastError());
}

}  // namespace pisces
