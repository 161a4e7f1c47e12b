// grad.hip -- the electron side of the analytic gradient on the grid.
//
// DVR::ComputeGradient (src/DVR.cpp:1099-1176) sums, over the grid points r_g
// with weights w_g = psi_g^2, the derivative of the potential with respect to
// every site position (Potential::EvaluateDPPGTOPGradient,
// src/Gradients.cpp:79-238; Potential 3, DampType 2, Polarization 3):
//   * the point charges, -q (dReff/dR) / Reff^2 along R / |R| (R = r - site);
//   * the Slater repulsive cores, -c zeta e^{-zeta R} along R / |R|;
//   * the electron's field E_i = g(R_i) R_i at the polarizable sites, whose
//     derivative dE_i/dR_i is dotted with the induced dipole mu_i of
//     mu = InvA (E + Epc) at that point (DerivElecField);
// and accumulates tmu = sum w mu and mcm = sum w mu mu^T (MuCrossMu), which the
// caller's water-side derivatives turn into the rest of the gradient
// (FinalGradient).  Here:
//   grad_sites_kernel: charges and cores;
//   grad_mu_kernel: mu of a tile of points on the matrix cores, then the dipole
//     terms and tmu per polarizable site;
//   grad_s_kernel: S = sum w (E + Epc)(E + Epc)^T on the matrix cores;
//   colsum_kernel, s_sum_kernel: partial sums added in a fixed order;
//   matmul_kernel: mcm = InvA S InvA.
// (H2O)24 on 64^3 (216 dimensions), us, before -> now: charges, cores and mu in
// one kernel 1633 -> 70 + 528, S 512 -> 333, sums 2 x 138 -> 9 + 2 x 5, products 2 x 60
// -> 2 x 11.  What was slow: 96 of 512 threads computing every exponential of a
// tile in series, the field's derivative per component instead of per site,
// 16-point tiles whose every step waited for memory and barriers, and one
// thread per column adding 1024 rows.  The matrix products alone take 0.34 ms (mu)
// and 0.17 ms (S) at the 72.7 TFLOP/s of a large FP64 product; 14 column blocks
// on 16 waves, the E rows and the site pass are the rest of mu, the E rows and
// two LDS operands per instruction that of S.
#include "common.hpp"
#include "context.hpp"
#include "gmem.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace pisces {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mma(double a, double b, f64x4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kLdsMax = 156 * 1024;  // E rows; the rest of a CU's LDS holds the points

struct GradDev {
    int nsites, np, n3p, pad;
    double qdamp, pdamp;
    const double *site4;  // per site: x, y, z, charge
    const double *srep;   // per site: zeta1, c1, zeta2, c2 (c = 0: unused)
    const double *rpol;   // 3 np: polarizable-site positions
    const double *epc;    // n3p: permanent-charge field (0 past 3 np)
    const double *inva;   // n3p x n3p, row-major, symmetric, zero-padded
};

struct GridDev {
    int nx, ny, nz;
    unsigned ng;
    const double *gx, *gy, *gz, *psi;
};

// effective distance, src/Potential.cpp:1191-1196, and dReff/dR
__device__ __forceinline__ double reff(double r, double r0, double &dre)
{
    if (r < r0) {
        const double t = r / r0;
        dre = 3.0 * t * t - 2.0 * t * t * t;
        return r0 * (0.5 + t * t * t * (1.0 - 0.5 * t));
    }
    dre = 1.0;
    return r;
}

// g(R) of the electron's field at a polarizable site (src/Gradients.cpp:131-142)
// from ri = 1/R; R2 > 0
__device__ __forceinline__ double field_g(double R2, double ri, double pdamp)
{
    const double R = R2 * ri;
    if (R < pdamp) {
        double dre;
        const double re = reff(R, pdamp, dre);
        return rcp64(re * re * re);
    }
    return ri * ri * ri;
}

// grid point g and its wavefunction value; past the grid the last point, with 0
__device__ __forceinline__ void point_of(const GridDev &G, unsigned g, double r[3], double &psi)
{
    const bool in = g < G.ng;
    const unsigned h = in ? g : G.ng - 1, iy = h / (unsigned)G.nx, iz = iy / (unsigned)G.ny;
    r[0] = G.gx[h - iy * G.nx];
    r[1] = G.gy[iy - iz * G.ny];
    r[2] = G.gz[iz];
    const double p = G.psi[h];
    psi = in ? p : 0.0;
}

// ------------------------------------------------------------------ charges and cores
// Bound by FP64 arithmetic (up to two exponentials a site and point).  A wave
// takes kSitesPerWave sites, its lanes the points of the workgroup's chunk, so
// that a point is decoded once for several sites and every lane computes; row
// blockIdx.x of part holds the chunk's 3 sums per site.
constexpr int kSitesNT = 512, kSitesPerWave = 4, kSitesChunk = 1024;

__global__ void __launch_bounds__(kSitesNT)
grad_sites_kernel(GradDev D, GridDev G, double *__restrict__ part)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s0 = (blockIdx.y * (kSitesNT / 64) + wave) * kSitesPerWave;
    if (s0 >= D.nsites) return;
    const cptr<double> s4 = cst(D.site4), sr = cst(D.srep);
    double f[kSitesPerWave][3];
#pragma unroll
    for (int k = 0; k < kSitesPerWave; ++k) f[k][0] = f[k][1] = f[k][2] = 0.0;
    for (int t = 0; t < kSitesChunk / 64; ++t) {
        const unsigned g = blockIdx.x * kSitesChunk + 64 * t + lane;
        double r[3], psi;
        point_of(G, g, r, psi);
        const double w = psi * psi;
#pragma unroll
        for (int k = 0; k < kSitesPerWave; ++k) {
            const int s = s0 + k;
            if (s >= D.nsites) break;
            const double rx = r[0] - s4[4 * s], ry = r[1] - s4[4 * s + 1], rz = r[2] - s4[4 * s + 2];
            const double q = s4[4 * s + 3], c1 = sr[4 * s + 1], c2 = sr[4 * s + 3];
            const double R2 = rx * rx + ry * ry + rz * rz;
            const bool on = w != 0.0 && R2 > 0.0;
            const double ri = rsq64(on ? R2 : 1.0), R = on ? R2 * ri : 1.0;
            double v = 0.0;  // dV/dR along R / |R|
            if (q != 0.0) {
                if (R < D.qdamp) {
                    double dre;
                    const double re = reff(R, D.qdamp, dre);
                    v -= q * dre / (re * re);
                } else {
                    v -= q * (ri * ri);
                }
            }
            if (c1 != 0.0) v += c1 * sr[4 * s] * exp(-sr[4 * s] * R);
            if (c2 != 0.0) v += c2 * sr[4 * s + 2] * exp(-sr[4 * s + 2] * R);
            const double fw = on ? w * v * ri : 0.0;
            f[k][0] += fw * rx;
            f[k][1] += fw * ry;
            f[k][2] += fw * rz;
        }
    }
#pragma unroll
    for (int k = 0; k < kSitesPerWave; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            double x = row_sum(f[k][a]);
            x += __shfl_xor(x, 16, 64);
            x += __shfl_xor(x, 32, 64);
            if (lane == 0 && s0 + k < D.nsites)
                part[(size_t)blockIdx.x * (3 * D.nsites) + 3 * (s0 + k) + a] = x;
        }
}

// ------------------------------------------------------------------ E rows
// Points of a tile (coordinates, psi) into pt, from the values a thread of the
// first PTS requested ahead.
struct PointReg {
    double r[3], psi;
};

// E rows (electron field + permanent-charge field) of PTS points in LDS, pitch
// n3p + 1 (odd: a column walk changes banks), zero past 3 np; SCALE: times psi.
template <int PTS, int NT, bool SCALE>
__device__ __forceinline__ void e_rows(const GradDev &D, const double (*pt)[4], double *Es)
{
    const int np = D.np, n3 = 3 * np, n3p = D.n3p, ldE = n3p + 1;
    const gptr<const double> rp = glb(D.rpol), ep = glb(D.epc);
    for (int idx = threadIdx.x; idx < PTS * np; idx += NT) {
        const int p = idx % PTS, i = idx / PTS;
        const double rx = pt[p][0] - rp[3 * i], ry = pt[p][1] - rp[3 * i + 1], rz = pt[p][2] - rp[3 * i + 2];
        const double R2 = rx * rx + ry * ry + rz * rz;
        const double g = R2 > 0.0 ? field_g(R2, rsq64(R2), D.pdamp) : 0.0;
        const double sc = SCALE ? pt[p][3] : 1.0;
        double *row = Es + p * ldE + 3 * i;
        row[0] = (g * rx + ep[3 * i]) * sc;
        row[1] = (g * ry + ep[3 * i + 1]) * sc;
        row[2] = (g * rz + ep[3 * i + 2]) * sc;
    }
    for (int idx = threadIdx.x; idx < PTS * (n3p - n3); idx += NT)
        Es[(idx % PTS) * ldE + n3 + idx / PTS] = 0.0;
}

// ------------------------------------------------------------------ induced dipoles
// mu = E InvA for tiles of 16 RB points, a workgroup walking the tiles t =
// blockIdx.x, + gridDim.x, ...: wave w computes the 16-column blocks w, w + NW,
// ... (ROUNDS at most) for all RB row blocks, InvA streamed from the L2 one
// k-group ahead; the dipoles then replace the E rows in LDS, and thread (sub, i)
// adds the terms of polarizable site i over the points p = sub, sub + nsub, ...:
//   F_a = w [(g'/R) (R . mu) R_a + g mu_a],  tmu = sum w mu.
// Bound by the FP64 matrix cores; the E rows and the site pass are about a
// quarter beside them.  Row blockIdx.x of part: 3 np tmu, 3 np forces.
constexpr int kMuNT = 1024;

template <int RB, int ROUNDS>
__global__ void __launch_bounds__(kMuNT)
grad_mu_kernel(GradDev D, GridDev G, unsigned ntiles, double *__restrict__ part)
{
    constexpr int PTS = 16 * RB, NW = kMuNT / 64;
    extern __shared__ double Es[];
    __shared__ double pt[PTS][4];
    const int n3p = D.n3p, ldE = n3p + 1, np = D.np, ncb = n3p / 16;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int sub = threadIdx.x / np, site = threadIdx.x - sub * np, nsub = kMuNT / np;
    const gptr<const double> A = glb(D.inva) + (lq * n3p + l16);
    double f[3] = {0.0, 0.0, 0.0}, tm[3] = {0.0, 0.0, 0.0}, sx = 0.0, sy = 0.0, sz = 0.0;
    if (sub < nsub) {
        sx = D.rpol[3 * site];
        sy = D.rpol[3 * site + 1];
        sz = D.rpol[3 * site + 2];
    }
    PointReg nx{};
    if (threadIdx.x < PTS) point_of(G, blockIdx.x * PTS + threadIdx.x, nx.r, nx.psi);
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (threadIdx.x < PTS) {
            pt[threadIdx.x][0] = nx.r[0];
            pt[threadIdx.x][1] = nx.r[1];
            pt[threadIdx.x][2] = nx.r[2];
            pt[threadIdx.x][3] = nx.psi;
            if (t + gridDim.x < ntiles) point_of(G, (t + gridDim.x) * PTS + threadIdx.x, nx.r, nx.psi);
        }
        __syncthreads();
        e_rows<PTS, kMuNT, false>(D, pt, Es);
        __syncthreads();
        f64x4 o[ROUNDS][RB];
        const double *ea = Es + l16 * ldE + lq;
#pragma unroll
        for (int u = 0; u < ROUNDS; ++u) {
#pragma unroll
            for (int b = 0; b < RB; ++b) o[u][b] = f64x4{0.0, 0.0, 0.0, 0.0};
            const int cb = wave + NW * u;
            if (cb >= ncb) break;
            const gptr<const double> bc = A + 16 * cb;
            double nv[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) nv[q] = bc[4 * q * n3p];
            for (int k0 = 0; k0 < n3p; k0 += 16) {
                double bv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) bv[q] = nv[q];
                const int kn = k0 + 16 < n3p ? k0 + 16 : 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) nv[q] = bc[(kn + 4 * q) * n3p];
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int b = 0; b < RB; ++b)
                        o[u][b] = mma(ea[16 * b * ldE + k0 + 4 * q], bv[q], o[u][b]);
            }
        }
        __syncthreads();  // every wave has read the E rows
#pragma unroll
        for (int u = 0; u < ROUNDS; ++u) {
            const int cb = wave + NW * u;
            if (cb >= ncb) break;
#pragma unroll
            for (int b = 0; b < RB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) Es[(16 * b + lq + 4 * r) * ldE + 16 * cb + l16] = o[u][b][r];
        }
        __syncthreads();
        if (sub < nsub)
            for (int p = sub; p < PTS; p += nsub) {
                const double w = pt[p][3] * pt[p][3];
                const double *m = Es + p * ldE + 3 * site;
                const double m0 = m[0], m1 = m[1], m2 = m[2];
                tm[0] += w * m0;
                tm[1] += w * m1;
                tm[2] += w * m2;
                const double rx = pt[p][0] - sx, ry = pt[p][1] - sy, rz = pt[p][2] - sz;
                const double R2 = rx * rx + ry * ry + rz * rz;
                if (R2 > 0.0) {
                    // g = Reff^-3, g'/R = -3 Reff' Reff^-4 / R (src/Gradients.cpp:187-198)
                    const double ri = rsq64(R2), R = R2 * ri;
                    double g = ri * ri * ri, dgr = -3.0 * g * ri * ri;
                    if (R < D.pdamp) {
                        double dre;
                        const double ire = rcp64(reff(R, D.pdamp, dre));
                        g = ire * ire * ire;
                        dgr = -3.0 * dre * (g * ire) * ri;
                    }
                    const double h = w * dgr * (rx * m0 + ry * m1 + rz * m2), gw = w * g;
                    f[0] += h * rx + gw * m0;
                    f[1] += h * ry + gw * m1;
                    f[2] += h * rz + gw * m2;
                }
            }
        __syncthreads();  // Es and pt are rewritten by the next tile
    }
    // the sub sums of each site, in order
    if (sub < nsub)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            Es[(sub * np + site) * 6 + a] = tm[a];
            Es[(sub * np + site) * 6 + 3 + a] = f[a];
        }
    __syncthreads();
    for (int e = threadIdx.x; e < 6 * np; e += kMuNT) {
        const int i = e / 6, a = e - 6 * i;
        double s = 0.0;
        for (int u = 0; u < nsub; ++u) s += Es[(u * np + i) * 6 + a];
        part[(size_t)blockIdx.x * (6 * np) + (a < 3 ? 3 * i + a : 3 * np + 3 * i + a - 3)] = s;
    }
}

// ------------------------------------------------------------------ S
// S = sum_p psi_p^2 (E_p + Epc)(E_p + Epc)^T = sum_p e_p e_p^T, e = psi (E +
// Epc), over its upper 16 x 16 blocks (bi <= bj, row by row) on the FP64 matrix
// cores.  blockIdx.y: a group of at most 16 kGradBPW blocks, split evenly over
// the waves; the workgroup walks the tiles of 16 RB points t = blockIdx.x, +
// gridDim.x, ..., builds their e rows in LDS, and each wave adds its blocks'
// products (k runs over the points) into register accumulators.  Partial:
// part[x][blk][16 x 16] row-major.
constexpr int kSNT = 1024, kGradBPW = 7;  // blocks per wave (8 registers each)

template <int RB>
__global__ void __launch_bounds__(kSNT)
grad_s_kernel(GradDev D, GridDev G, unsigned ntiles, int blk_per_grp, double *__restrict__ part)
{
    constexpr int PTS = 16 * RB, NW = kSNT / 64;
    extern __shared__ double Es[];
    __shared__ double pt[PTS][4];
    const int n3p = D.n3p, ldE = n3p + 1;
    const int ncb = n3p / 16, nblk = ncb * (ncb + 1) / 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    // this wave's blocks: a contiguous run of the group's
    const int g0 = blockIdx.y * blk_per_grp, gn = nblk - g0 < blk_per_grp ? nblk - g0 : blk_per_grp;
    const int b0 = g0 + gn * wave / NW, nown = g0 + gn * (wave + 1) / NW - b0;
    int oa[kGradBPW], ob[kGradBPW];
    {
        int bi = 0, bj = b0;
        while (bi < ncb && bj >= ncb - bi) {
            bj -= ncb - bi;
            ++bi;
        }
        bj += bi;
#pragma unroll
        for (int u = 0; u < kGradBPW; ++u) {
            oa[u] = 16 * bi;
            ob[u] = 16 * bj;
            if (++bj == ncb) bj = ++bi;
        }
    }
    f64x4 acc[kGradBPW];
#pragma unroll
    for (int u = 0; u < kGradBPW; ++u) acc[u] = f64x4{0.0, 0.0, 0.0, 0.0};
    PointReg nx{};
    if (threadIdx.x < PTS) point_of(G, blockIdx.x * PTS + threadIdx.x, nx.r, nx.psi);
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (threadIdx.x < PTS) {
            pt[threadIdx.x][0] = nx.r[0];
            pt[threadIdx.x][1] = nx.r[1];
            pt[threadIdx.x][2] = nx.r[2];
            pt[threadIdx.x][3] = nx.psi;
            if (t + gridDim.x < ntiles) point_of(G, (t + gridDim.x) * PTS + threadIdx.x, nx.r, nx.psi);
        }
        __syncthreads();
        e_rows<PTS, kSNT, true>(D, pt, Es);
        __syncthreads();
        // k-step q: points 4 q + lq; A[c1][k] = e[4 q + k][16 bi + c1], B[k][c2] = e[..][16 bj + c2]
#pragma unroll 1
        for (int q = 0; q < PTS / 4; ++q) {
            const double *e = Es + (4 * q + lq) * ldE + l16;
#pragma unroll
            for (int u = 0; u < kGradBPW; ++u)
                if (u < nown) acc[u] = mma(e[oa[u]], e[ob[u]], acc[u]);
        }
        __syncthreads();  // Es and pt are rewritten by the next tile
    }
#pragma unroll
    for (int u = 0; u < kGradBPW; ++u) {
        if (u >= nown) break;
        double *out = part + ((size_t)blockIdx.x * nblk + b0 + u) * 256;
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(lq + 4 * r) * 16 + l16] = acc[u][r];
    }
}

// ------------------------------------------------------------------ sums
// Sum over the rows of part[row][c] of 64 columns per workgroup: 16 threads a
// column add every 16th row, then the 16 sums in order.
constexpr int kSumSplit = 16;

__device__ __forceinline__ double col_sum(const double *__restrict__ part, int rows, long long cols,
                                          long long c, bool in, double (*red)[64])
{
    const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (in) {
        int r = q;
        for (; r + 3 * kSumSplit < rows; r += 4 * kSumSplit)
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += part[(long long)(r + u * kSumSplit) * cols + c];
        for (; r < rows; r += kSumSplit) s[0] += part[(long long)r * cols + c];
    }
    red[q][lane] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    double t = 0.0;
    if (q == 0)
#pragma unroll
        for (int u = 0; u < kSumSplit; ++u) t += red[u][lane];
    return t;
}

__global__ void __launch_bounds__(64 * kSumSplit)
colsum_kernel(const double *__restrict__ part, int rows, long long cols, double *__restrict__ out)
{
    __shared__ double red[kSumSplit][64];
    const long long c = (long long)blockIdx.x * 64 + (threadIdx.x & 63);
    const double t = col_sum(part, rows, cols, c, c < cols, red);
    if (threadIdx.x < 64 && c < cols) out[c] = t;
}

// The block sums of S, into both triangles of the n3p x n3p matrix.
__global__ void __launch_bounds__(64 * kSumSplit)
s_sum_kernel(const double *__restrict__ part, int rows, int n3p, double *__restrict__ S)
{
    __shared__ double red[kSumSplit][64];
    const int ncb = n3p / 16, nblk = ncb * (ncb + 1) / 2;
    const long long c = (long long)blockIdx.x * 64 + (threadIdx.x & 63);  // nblk * 256 columns
    const double t = col_sum(part, rows, (long long)nblk * 256, c, true, red);
    if (threadIdx.x >= 64) return;
    int bj = (int)(c >> 8), bi = 0;
    while (bj >= ncb - bi) {
        bj -= ncb - bi;
        ++bi;
    }
    bj += bi;
    const int r = 16 * bi + ((int)(c >> 4) & 15), k = 16 * bj + ((int)c & 15);
    if (bi == bj && r > k) return;  // the diagonal blocks' upper halves serve both
    S[(size_t)r * n3p + k] = t;
    S[(size_t)k * n3p + r] = t;
}

// The leading nc x nc part of C = A B (pitch nc) for n x n row-major matrices (n a
// multiple of 16), a wave per 16 x 16 tile, four 16-wide k-groups in flight.
__global__ void __launch_bounds__(256)
matmul_kernel(const double *__restrict__ A_, const double *__restrict__ B_, int n, double *__restrict__ C,
              int nc)
{
    const int nb = n / 16, tile = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (tile >= nb * nb) return;
    const int ti = tile / nb, tj = tile - ti * nb;
    const int l16 = threadIdx.x & 15, lq = (threadIdx.x & 63) >> 4;
    const gptr<const double> A = glb(A_) + (16 * ti + l16) * n + lq, B = glb(B_) + lq * n + 16 * tj + l16;
    f64x4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll 4
    for (int k0 = 0; k0 < n; k0 += 16)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q & 1] = mma(A[k0 + 4 * q], B[(k0 + 4 * q) * n], acc[q & 1]);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (16 * ti + lq + 4 * r < nc && 16 * tj + l16 < nc)
            C[(size_t)(16 * ti + lq + 4 * r) * nc + 16 * tj + l16] = acc[0][r] + acc[1][r];
}

template <typename K> void allow_lds(K kernel)
{
    PC_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax));
}

}  // namespace

void gradient_terms(pisces_ctx *c, const double *psi_host, double *gel, double *tmu, double *mcm)
{
    GradState &G = c->gs;
    PC_REQUIRE(G.valid, PISCES_ERR_STATE,
               "the gradient needs a PolType 3 potential (Potential 3, DampType 2, Polarization 3) "
               "built on this context");
    const int ns = G.nsites, np = G.np, n3p = G.n3p, n3 = 3 * np, ncb = n3p / 16;
    const unsigned ng = (unsigned)c->ngp;
    static std::once_flag once;
    std::call_once(once, [] {
        allow_lds(grad_mu_kernel<4, 1>);
        allow_lds(grad_mu_kernel<2, 2>);
        allow_lds(grad_mu_kernel<2, 3>);
        allow_lds(grad_s_kernel<4>);
        allow_lds(grad_s_kernel<2>);
    });
    // 64-point tiles up to one column block per wave (their E rows then fit the
    // LDS), else 32
    const size_t row = (size_t)(n3p + 1) * sizeof(double);
    const int rb = ncb <= kMuNT / 64 ? 4 : 2, pts = 16 * rb;
    const size_t lds = std::max(pts * row, (size_t)kMuNT * 6 * sizeof(double));
    PC_REQUIRE(lds <= (size_t)kLdsMax && n3p <= kPol3MaxN, PISCES_ERR_UNSUPPORTED,
               "too many polarizable sites for the gradient");
    PC_REQUIRE(ns <= 1024, PISCES_ERR_UNSUPPORTED, "too many sites for the gradient");
    GradDev D{ns, np, n3p, 0, G.qdamp, G.pdamp, G.site4.as<double>(), G.srep.as<double>(),
              G.rpol.as<double>(), G.epc.as<double>(), G.inva.as<double>()};
    const unsigned ntiles = (ng + pts - 1) / pts;
    const int nblk = ncb * (ncb + 1) / 2;
    const int chunks = (int)((ng + kSitesChunk - 1) / kSitesChunk);
    // one workgroup per CU for each of the two matrix-core kernels
    const int wg = (int)std::min<unsigned>(ntiles, 256);
    const int ngrp = (nblk + 16 * kGradBPW - 1) / (16 * kGradBPW), bpg = (nblk + ngrp - 1) / ngrp;
    const int nk = (int)std::min<unsigned>(ntiles, std::max(1, 256 / ngrp));
    const long long nn = (long long)n3p * n3p, cmu = 6LL * np;
    // workspace of the context: psi, the partial sums, their sums, S and two products
    size_t off = 0;
    auto take = [&](size_t doubles) {
        const size_t o = off;
        off += (doubles + 31) & ~(size_t)31;
        return o;
    };
    const size_t o_psi = take(ng), o_sites = take((size_t)chunks * 3 * ns), o_mu = take((size_t)wg * cmu),
                 o_s = take((size_t)nk * nblk * 256), o_tot = take(3 * ns + cmu), o_S = take(nn),
                 o_T = take(nn), o_M = take(nn);
    c->wgrad.ensure(off * sizeof(double));
    double *w = c->wgrad.as<double>();
    GridDev R{c->n[0], c->n[1], c->n[2], ng, c->dx[0].as<double>(), c->dx[1].as<double>(),
              c->dx[2].as<double>(), w + o_psi};
    hipStream_t s = c->stream;
    PC_HIP(hipMemcpyAsync(w + o_psi, psi_host, sizeof(double) * ng, hipMemcpyHostToDevice, s));
    auto go = [&](auto s_kernel, auto mu_kernel) {
        hipLaunchKernelGGL(s_kernel, dim3(nk, ngrp), dim3(kSNT), pts * row, s, D, R, ntiles, bpg, w + o_s);
        hipLaunchKernelGGL(mu_kernel, dim3(wg), dim3(kMuNT), lds, s, D, R, ntiles, w + o_mu);
    };
    if (rb == 4) go(grad_s_kernel<4>, grad_mu_kernel<4, 1>);
    else if (ncb <= 2 * (kMuNT / 64)) go(grad_s_kernel<2>, grad_mu_kernel<2, 2>);
    else go(grad_s_kernel<2>, grad_mu_kernel<2, 3>);
    const int sg = (ns + kSitesPerWave * (kSitesNT / 64) - 1) / (kSitesPerWave * (kSitesNT / 64));
    hipLaunchKernelGGL(grad_sites_kernel, dim3(chunks, sg), dim3(kSitesNT), 0, s, D, R, w + o_sites);
    const dim3 sb(64 * kSumSplit);
    hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((3 * ns + 63) / 64)), sb, 0, s, w + o_sites, chunks,
                       (long long)3 * ns, w + o_tot);
    hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)((cmu + 63) / 64)), sb, 0, s, w + o_mu, wg, cmu,
                       w + o_tot + 3 * ns);
    hipLaunchKernelGGL(s_sum_kernel, dim3((unsigned)(nblk * 4)), sb, 0, s, w + o_s, nk, n3p, w + o_S);
    // mcm = InvA S InvA
    const unsigned mb = (unsigned)((ncb * ncb + 3) / 4);
    hipLaunchKernelGGL(matmul_kernel, dim3(mb), dim3(256), 0, s, w + o_S, G.inva.as<double>(), n3p, w + o_T, n3p);
    hipLaunchKernelGGL(matmul_kernel, dim3(mb), dim3(256), 0, s, G.inva.as<double>(), w + o_T, n3p, w + o_M, n3);
    PC_HIP(hipGetLastError());
    std::vector<double> tot(3 * ns + cmu);
    PC_HIP(hipMemcpyAsync(tot.data(), w + o_tot, sizeof(double) * tot.size(), hipMemcpyDeviceToHost, s));
    PC_HIP(hipMemcpyAsync(mcm, w + o_M, sizeof(double) * n3 * n3, hipMemcpyDeviceToHost, s));
    c->sync();
    for (int k = 0; k < 3 * ns; ++k) gel[k] = tot[k];
    const double *f = tot.data() + 3 * ns + n3;
    for (int i = 0; i < np; ++i)
        for (int a = 0; a < 3; ++a) gel[3 * G.ip[i] + a] += f[3 * i + a];
    for (int k = 0; k < n3; ++k) tmu[k] = tot[3 * ns + k];
}

}  // namespace pisces
