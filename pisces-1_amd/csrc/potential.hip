// potential.hip -- electron-water potential on the grid, and the FP64 induced-
// dipole solve of the water model, for gfx950.
//
// Grid build: DVR::ComputePotential with sampling 1 (src/DVR.cpp:661-859) calls
// Potential::Evaluate (src/Potential.cpp:128-182) -> EvaluateDPPGTOP (:844-956)
// at every grid point.  The work is N_grid x N_site FP64 arithmetic, compute-bound
// on the FP64 VALU: a reciprocal square root per distance (1/R to ~1 ulp; R, R^-3,
// R^-4 follow by products, exact divisions only inside the damping radii) and one
// exp per repulsive core.  So the cluster's lists are merged by site on the host
// (a water's three charges, three dipoles, four cores and one polarizability sit
// on four sites: four distances instead of eleven), a thread of a large launch
// takes two points of one column, which share x, y and the entry's loads, and the
// entries are read as scalar loads through the constant address space.  The
// per-site distance table of the reference (Rx, Ry, Rz, R2, R, Rminus3;
// src/Potential.cpp:136-146) is recomputed instead of stored, with expressions
// that agree with it to rounding.
#include "common.hpp"
#include "gmem.hpp"

#include <algorithm>
#include <mutex>

namespace pisces {

namespace {

constexpr int kPotThreads = 256;
constexpr int kMaxSites = 1024;
// Points of a thread: 2 from kPotTwo points a launch on, 1 below, where the waves
// would be too few to cover the entries' loads.  us, 1 / 2 points, at 8, 24 and 45
// waters: 64^3 (262144 points) 26.4 / 28.4, 70.2 / 75.9, 126 / 132; 72 x 64^2
// (294912) 30.5 / 30.8, 80.4 / 81.7, 145 / 147; 72^3 (373248) 34.8 / 32.0, 92.3 /
// 83.9, 167 / 152; 80^3 (512000) 44.6 / 38.4, 119 / 103, 214 / 186; 96^3 70.0 /
// 59.3, 194 / 164, 354 / 295; 32 grids of 24 waters 64^3 in one launch 1590 / 1279.
// Four points at 64^3, 96^3 and the 32 grids: 97, 273, 1269.  (Eleven distances a
// water and one point: 98, 358, 2505.)
constexpr long long kPotTwo = 327680;
int pot_points(long long points) { return points >= kPotTwo ? 2 : 1; }

__device__ inline double reff(double r, double r0)
{
    // effective-distance damping, src/Potential.cpp:1191-1196
    if (r < r0) {
        const double t = r / r0;
        return r0 * (0.5 + t * t * t * (1.0 - 0.5 * t));
    }
    return r;
}

// |r| from r^2 and 1/|r| (0 at r = 0, where 1/|r| is infinite)
__device__ __forceinline__ double norm_of(double r2, double ri) { return r2 > 0.0 ? r2 * ri : 0.0; }

// Thread t of a grid: the points (i, j, k), (i, j, k + zh), ... of a column,
// zh = ceil(nz / K).
template <int DAMP, int K>
__device__ __forceinline__ void potential_points(const PotParams &P, const PotDev &D, int nx, int ny, int nz,
                                 const double *__restrict__ gx, const double *__restrict__ gy,
                                 const double *__restrict__ gz, double *__restrict__ v,
                                 float *__restrict__ v32, long long t)
{
    const int zh = (nz + K - 1) / K;
    const long long nxy = (long long)nx * ny;
    if (t >= nxy * zh) return;
    int i, j, k0;
    if (nxy * zh <= 0x7fffffff) {  // 32-bit divisions; uniform
        const unsigned u = (unsigned)t, w = u / (unsigned)nx;
        i = (int)(u - w * (unsigned)nx);
        k0 = (int)(w / (unsigned)ny);
        j = (int)(w - (unsigned)k0 * (unsigned)ny);
    } else {
        const long long w = t / nx;
        i = (int)(t - w * nx);
        k0 = (int)(w / ny);
        j = (int)(w - (long long)k0 * ny);
    }
    const double r0 = gx[i], r1 = gy[j];
    double r2[K];
#pragma unroll
    for (int p = 0; p < K; ++p) r2[p] = gz[min(k0 + p * zh, nz - 1)];
    const cptr<double> ionx = cst(D.ion_xyz), ionq = cst(D.ion_q);
    const cptr<PotSite> ent = cst(D.ent);
    const cptr<double> dm = cst(D.d), rp = cst(D.rep);
    double vpc[K] = {}, vind[K] = {}, vrep[K] = {}, sp[K] = {};
    const double qd2 = P.qdamp * P.qdamp, dd2 = P.ddamp * P.ddamp, pd2 = P.pdamp * P.pdamp;
    for (int c = 0; c < D.nent; ++c) {
        const cptr<PotSite> ep = ent + c;
        const PotSite e{ep->x, ep->y, ep->z, ep->q, ep->dip, ep->r0, ep->r1, ep->pol};
        const double ez = e.z, eq = e.q;
        const int dip = e.dip, c0 = e.r0, c1 = e.r1, pol = e.pol;
        const double rx = r0 - e.x, ry = r1 - e.y, rxy = rx * rx + ry * ry;
        double rz[K], R2[K], ri[K];
#pragma unroll
        for (int p = 0; p < K; ++p) {
            rz[p] = r2[p] - ez;
            R2[p] = fma(rz[p], rz[p], rxy);
            ri[p] = rsq64(R2[p]);
        }
        // point charge, src/Potential.cpp:1168-1210
        if (eq != 0.0) {
#pragma unroll
            for (int p = 0; p < K; ++p) {
                if (DAMP == 1) {
                    vpc[p] += -eq * ri[p] * (1.0 - exp(-P.qdamp * R2[p]));
                } else {
                    double u = ri[p];
                    if (R2[p] < qd2) u = 1.0 / reff(norm_of(R2[p], ri[p]), P.qdamp);
                    vpc[p] = fma(-eq, u, vpc[p]);
                }
            }
        }
        // point dipole, src/Potential.cpp:1222-1270
        if (dip >= 0) {
            const double dz = dm[3 * dip + 2], dxy = rx * dm[3 * dip] + ry * dm[3 * dip + 1];
#pragma unroll
            for (int p = 0; p < K; ++p) {
                const double dot = fma(rz[p], dz, dxy);
                double rm3 = ri[p] * ri[p] * ri[p];
                if (DAMP == 1) {
                    const double dd = 1.0 - exp(-P.ddamp * R2[p]);
                    vind[p] += -dot * rm3 * dd * dd;
                } else {
                    if (R2[p] < dd2) {
                        const double re = reff(norm_of(R2[p], ri[p]), P.ddamp);
                        rm3 = 1.0 / (re * re * re);
                    }
                    vind[p] = fma(-dot, rm3, vind[p]);
                }
            }
        }
        // repulsive cores, src/Potential.cpp:1282-1315
        for (int r = c0; r < c1; ++r) {
            const double ea = rp[2 * r], ef = rp[2 * r + 1];
#pragma unroll
            for (int p = 0; p < K; ++p)
                vrep[p] = fma(ef, exp(-ea * (P.rep_type == 1 ? R2[p] : norm_of(R2[p], ri[p]))), vrep[p]);
        }
        // polarization of a non-interacting site, src/Potential.cpp:1331-1374, :875-887
        if (pol) {
#pragma unroll
            for (int p = 0; p < K; ++p) {
                const double ri2 = ri[p] * ri[p];
                double u = ri2 * ri2;
                if (DAMP == 1) {
                    const double dd = 1.0 - exp(-P.pdamp * R2[p]);
                    u *= dd * dd;
                } else if (R2[p] < pd2) {
                    const double re = reff(norm_of(R2[p], ri[p]), P.pdamp), re2 = re * re;
                    u = R2[p] / (re2 * re2 * re2);
                }
                sp[p] = fma(P.alpha, u, sp[p]);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < K; ++p) {
        const int k = k0 + p * zh;
        if (k >= nz) break;
        double vt = vpc[p] + vind[p] + vrep[p];
        if (P.pol_type == 1) vt += P.adiabatic ? P.eps - sqrt(P.eps * (P.eps + sp[p])) : -0.5 * sp[p];
        // ions: erf-damped charges (Bloomfield form, src/NaCl.cpp:300-307)
        for (int c = 0; c < D.nion; ++c) {
            const double rx = r0 - ionx[3 * c], ry = r1 - ionx[3 * c + 1], rz = r2[p] - ionx[3 * c + 2];
            const double R2 = rx * rx + ry * ry + rz * rz;
            const double ri = rsq64(R2);
            vt += -ionq[c] * erf(norm_of(R2, ri) / P.ion_r) * ri;
        }
        const long long g = i + (long long)nx * j + nxy * k;
        if (v) v[g] = vt;
        if (v32) v32[g] = (float)vt;
    }
}

template <int K>
__global__ void __launch_bounds__(kPotThreads)
potential_grid_kernel(PotParams P, PotDev D, int nx, int ny, int nz, const double *__restrict__ gx,
                      const double *__restrict__ gy, const double *__restrict__ gz,
                      double *__restrict__ v, float *__restrict__ v32)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (P.damp_type == 1) potential_points<1, K>(P, D, nx, ny, nz, gx, gy, gz, v, v32, t);
    else potential_points<2, K>(P, D, nx, ny, nz, gx, gy, gz, v, v32, t);
}

// many clusters in one launch: blockIdx.y selects the task
template <int K>
__global__ void __launch_bounds__(kPotThreads)
potential_grid_batched_kernel(PotParams P, const PotTask *__restrict__ tasks)
{
    const PotTask &q = tasks[blockIdx.y];
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (P.damp_type == 1) potential_points<1, K>(P, q.D, q.nx, q.ny, q.nz, q.gx, q.gy, q.gz, q.v, q.v32, t);
    else potential_points<2, K>(P, q.D, q.nx, q.ny, q.nz, q.gx, q.gy, q.gz, q.v, q.v32, t);
}

// --------------------------------------------------------------------------
// Induced dipoles of the rigid DPP waters, FP64, one workgroup per cluster.
// WaterCluster::CalcInducedDipoles (src/DPP.cpp:760-1065): field of the
// permanent charges of the other waters at the polarizable sites (O, H1, H2),
// then the 0.5-mixed fixed-point iteration mu <- 0.5 mu + 0.5 alpha (E_pc +
// T mu) until the mean change drops below 1e-12.  The damped dipole tensor of a
// pair (src/DPP.cpp:2377-2410) is T = a r r^T - b, a = 3 d1 / r^5, b = d2 / r^3,
// and does not change during the iteration: each thread computes a and b of its
// pairs once and keeps them in registers.
//
// The iteration is a serial chain of some fifty small steps on one CU, so its
// cost is the length of a step.  The threads are split evenly over
// the sites, 2^lg lanes of one wave per site; a lane sums its partners j = part,
// part + 2^lg, ..., the lanes' sums meet by lane permutes, dipoles and the
// waves' shares of the change are double-buffered in LDS, and every thread adds
// those shares itself: one barrier per step.  A thread's first HELD pairs (all of
// them up to 24 waters) stay in registers, as sqrt(a) r and b, which
// leaves only the partner's dipole to read; of the rest, (a, b) of as many as
// fit are kept in LDS and the remainder in `work`, laid out so that a wave reads
// it contiguously.  us a launch, before (6-element tensors from global memory,
// 256 threads, ten barriers a step) -> now: 24 waters 427 -> 91, 45 waters
// 1834 -> 313.
//
// Two forms: 640 threads (three waves a SIMD, so that nine pairs fit the
// registers; twelve spilled) up to 640 sites, 1024 threads (six pairs) beyond.
template <int NT> struct Scf {
    static constexpr int HELD = NT == 640 ? 9 : 6;      // pairs of a thread in registers
    static constexpr int SLOT_BYTES = NT * 2 * (int)sizeof(double);
    static constexpr int LDS = 152 * 1024;
    // lanes per site, as a power of two: the most that fit
    __host__ __device__ static int lg(int ns)
    {
        int l = 6;
        while (l > 0 && (ns << l) > NT) --l;
        return l;
    }
    __host__ __device__ static int pairs(int ns) { return (ns + (1 << lg(ns)) - 1) >> lg(ns); }
    // pairs of a thread in LDS, beside the 9 ns doubles of positions and dipoles
    __host__ __device__ static int slots(int ns)
    {
        const int left = (LDS - 8 * (9 * ns + 1)) / SLOT_BYTES, want = pairs(ns) - HELD;
        return want < 0 ? 0 : want < left ? want : left;
    }
};
constexpr int kScfSmall = 640, kScfLarge = 1024;
// the form of a cluster of ns sites: its order of summation, so never that of
// another cluster of the launch
__host__ __device__ inline int scf_threads(int ns) { return ns <= kScfSmall ? kScfSmall : kScfLarge; }
constexpr double kA2B = 1.0 / 0.52917720859;
constexpr double kPolO = 1.22 * kA2B * kA2B * kA2B, kPolH = 0.28 * kA2B * kA2B * kA2B;

// Sums over groups of 2^to lanes whose sub-groups of 2^from lanes hold equal
// values: xor 1, 2 by DPP quad permutes, then (equal groups of 4 and 8) the half
// row and row mirrors, then shuffles.
__device__ __forceinline__ double scf_lanes(double x, int from, int to)
{
    if (from <= 0 && to > 0) x = dpp_add<0xB1>(x);
    if (from <= 1 && to > 1) x = dpp_add<0x4E>(x);
    if (from <= 2 && to > 2) x = dpp_add<0x141>(x);
    if (from <= 3 && to > 3) x = dpp_add<0x140>(x);
    if (from <= 4 && to > 4) x += __shfl_xor(x, 16, 64);
    if (from <= 5 && to > 5) x += __shfl_xor(x, 32, 64);
    return x;
}

// polarizabilities (O, H1, H2), charges (H1, H2, M) and the charges' damping
// polarizabilities: src/Water.cpp:233-236 (chargeselector 2) with
// src/ttm_data.h:14-15, 51-52
__device__ __forceinline__ double scf_alpha(int i) { return i % 3 == 0 ? kPolO : kPolH; }
// 1 / sqrt(alpha alpha') of two sites by how many of them are oxygens (or M for
// a charge): sqrt(1.22 * 0.28)
constexpr double kSqrtOH = 0.58446556784809830;
__device__ __forceinline__ double scf_damp_scale(int oxygens)
{
    constexpr double a3 = kA2B * kA2B * kA2B;
    return oxygens == 2 ? 1.0 / kPolO : oxygens == 1 ? 1.0 / (kSqrtOH * a3) : 1.0 / kPolH;
}

template <int NT>
__device__ __forceinline__ void water_scf_body(int nw, const double *__restrict__ sites, double *__restrict__ mu_out,
                               double *__restrict__ epc_out, double *__restrict__ work,
                               int *__restrict__ info)
{
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    const double dampCD = 0.21, dampDD = 0.3;  // src/Water.cpp:243
    const double qH = 0.5742185854046506;
    constexpr int HELD = Scf<NT>::HELD;
    const int ns = 3 * nw, lg = Scf<NT>::lg(ns), nu = Scf<NT>::pairs(ns);
    // positions, two sets of dipoles (3 ns each), then the LDS pairs
    extern __shared__ __align__(16) double scf_lds[];
    __shared__ double red[2][NT / 64];
    double *px = scf_lds, *m0 = scf_lds + 3 * ns;
    f64x2 *slot = reinterpret_cast<f64x2 *>(scf_lds + 9 * ns + (ns & 1));
    const int nslot = Scf<NT>::slots(ns), first = HELD + nslot;  // first pair in `work`
    const int tid = threadIdx.x;
    const int i = tid >> lg, part = tid & ((1 << lg) - 1);
    const bool own = i < ns;
    for (int k = tid; k < 3 * ns; k += NT) {
        const int s = k / 3;
        px[k] = sites[12 * (s / 3) + 3 * (s % 3) + k % 3];
    }
    __syncthreads();
    const double ai = own ? scf_alpha(i) : 0.0;
    const double xi = own ? px[3 * i] : 0.0, yi = own ? px[3 * i + 1] : 0.0, zi = own ? px[3 * i + 2] : 0.0;
    // pair coefficients
    auto pair = [&](int j) {
        f64x2 c = {0.0, 0.0};
        if (own && j < ns && j != i) {
            const double rx = xi - px[3 * j], ry = yi - px[3 * j + 1], rz = zi - px[3 * j + 2];
            const double r2 = rx * rx + ry * ry + rz * rz, ri = rsq64(r2), ri3 = ri * ri * ri;
            const double x = dampDD * (r2 * r2 * ri) * scf_damp_scale((i % 3 == 0) + (j % 3 == 0)), ex = exp(-x);
            c[0] = 3.0 * (1.0 - (1.0 + x) * ex) * ri3 * ri * ri;
            c[1] = (1.0 - ex) * ri3;
        }
        return c;
    };
    double sx[HELD], sy[HELD], sz[HELD], sb[HELD];
#pragma unroll
    for (int u = 0; u < HELD; ++u) {
        const int j = part + (u << lg), jj = j < ns ? j : 0;
        const f64x2 c = pair(j);
        // a is the rounding of its factor, either sign, between sites that nearly coincide
        const double sa = sqrt(c[0] < 0.0 ? 0.0 : c[0]);
        sx[u] = sa * (xi - px[3 * jj]);
        sy[u] = sa * (yi - px[3 * jj + 1]);
        sz[u] = sa * (zi - px[3 * jj + 2]);
        sb[u] = c[1];
        __builtin_amdgcn_sched_barrier(0);  // one pair's temporaries at a time
    }
    f64x2 *rest = reinterpret_cast<f64x2 *>(work) + tid;
    for (int u = 0; u < nslot; ++u) slot[u * NT + tid] = pair(part + ((HELD + u) << lg));
    for (int u = first; u < nu; ++u) rest[(size_t)(u - first) * NT] = pair(part + (u << lg));
    // permanent-charge field (src/DPP.cpp:830-865)
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;
    for (int q = part; q < 3 * nw; q += 1 << lg) {
        const int w = q / 3, s = 1 + q % 3;  // H1, H2, M of water w
        if (!own || i / 3 == w) continue;
        const double *pc = sites + 12 * w + 3 * s;
        const double rx = xi - pc[0], ry = yi - pc[1], rz = zi - pc[2];
        const double r2 = rx * rx + ry * ry + rz * rz, ri = rsq64(r2);
        const double x = dampCD * (r2 * r2 * ri) * scf_damp_scale((i % 3 == 0) + (s == 3));
        const double t = (s == 3 ? -2.0 * qH : qH) * ri * ri * ri * (1.0 - exp(-x));
        f0 += t * rx;
        f1 += t * ry;
        f2 += t * rz;
    }
    f0 = scf_lanes(f0, 0, lg);
    f1 = scf_lanes(f1, 0, lg);
    f2 = scf_lanes(f2, 0, lg);
    double o0 = 0.5 * ai * f0, o1 = 0.5 * ai * f1, o2 = 0.5 * ai * f2;
    if (own && part == 0) {
        epc_out[3 * i] = f0;
        epc_out[3 * i + 1] = f1;
        epc_out[3 * i + 2] = f2;
        m0[3 * i] = o0;
        m0[3 * i + 1] = o1;
        m0[3 * i + 2] = o2;
    }
    __syncthreads();
    const int maxit = 5 * (ns + 10);
    const double tol2 = (3e-12 * ns) * (3e-12 * ns);  // |change| / 3 / ns < 1e-12
    int it = 0, conv = 0;
    for (it = 0; it < maxit; ++it) {
        const double *cur = m0 + 3 * ns * (it & 1);
        double *nxt = m0 + 3 * ns * ((it & 1) ^ 1);
        double e0 = 0.0, e1 = 0.0, e2 = 0.0;
        auto add = [&](int j, f64x2 c) {
            const int jj = j < ns ? j : 0;  // c = 0 past the last site
            const double u0 = cur[3 * jj], u1 = cur[3 * jj + 1], u2 = cur[3 * jj + 2];
            const double rx = xi - px[3 * jj], ry = yi - px[3 * jj + 1], rz = zi - px[3 * jj + 2];
            const double d = c[0] * (rx * u0 + ry * u1 + rz * u2);
            e0 += d * rx - c[1] * u0;
            e1 += d * ry - c[1] * u1;
            e2 += d * rz - c[1] * u2;
        };
        if (own) {
#pragma unroll
            for (int u = 0; u < HELD; ++u)
                if (u < nu) {
                    const int j = part + (u << lg), jj = j < ns ? j : 0;
                    const double u0 = cur[3 * jj], u1 = cur[3 * jj + 1], u2 = cur[3 * jj + 2];
                    const double d = sx[u] * u0 + sy[u] * u1 + sz[u] * u2;
                    e0 += d * sx[u] - sb[u] * u0;
                    e1 += d * sy[u] - sb[u] * u1;
                    e2 += d * sz[u] - sb[u] * u2;
                }
            for (int u = 0; u < nslot; ++u) add(part + ((HELD + u) << lg), slot[u * NT + tid]);
#pragma unroll 4
            for (int u = first; u < nu; ++u) add(part + (u << lg), rest[(size_t)(u - first) * NT]);
        }
        e0 = scf_lanes(e0, 0, lg);
        e1 = scf_lanes(e1, 0, lg);
        e2 = scf_lanes(e2, 0, lg);
        const double n0 = 0.5 * o0 + 0.5 * ai * (f0 + e0);
        const double n1 = 0.5 * o1 + 0.5 * ai * (f1 + e1);
        const double n2 = 0.5 * o2 + 0.5 * ai * (f2 + e2);
        // the lanes of a site hold the same change: sum over the wave's sites
        double d = (o0 - n0) * (o0 - n0) + (o1 - n1) * (o1 - n1) + (o2 - n2) * (o2 - n2);
        d = scf_lanes(own ? d : 0.0, lg, 6);
        if (own && part == 0) {
            nxt[3 * i] = n0;
            nxt[3 * i + 1] = n1;
            nxt[3 * i + 2] = n2;
        }
        o0 = n0;
        o1 = n1;
        o2 = n2;
        if ((tid & 63) == 0) red[it & 1][tid >> 6] = d;
        __syncthreads();  // the new dipoles and every wave's share are in LDS
        double s2[2] = {0.0, 0.0};
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) s2[w & 1] += red[it & 1][w];
        if (s2[0] + s2[1] < tol2) {
            conv = 1;
            break;
        }
    }
    if (own && part == 0) {
        mu_out[3 * i] = o0;
        mu_out[3 * i + 1] = o1;
        mu_out[3 * i + 2] = o2;
    }
    if (tid == 0) {
        info[0] = conv;
        info[1] = conv ? it + 1 : it;
    }
}

template <int NT>
__global__ void __launch_bounds__(NT)
water_scf_kernel(int nw, const double *__restrict__ sites, double *__restrict__ mu_out,
                 double *__restrict__ epc_out, double *__restrict__ work, int *__restrict__ info)
{
    water_scf_body<NT>(nw, sites, mu_out, epc_out, work, info);
}

// one cluster per workgroup; clusters of the other form are left to its launch
template <int NT>
__global__ void __launch_bounds__(NT) water_scf_batched_kernel(const ScfTask *__restrict__ tasks)
{
    const ScfTask &t = tasks[blockIdx.x];
    if (scf_threads(3 * t.nw) != NT) return;
    water_scf_body<NT>(t.nw, t.sites, t.mu, t.epc, t.work, t.info);
}

}  // namespace

void potential_grid_launch(const PotParams &P, const PotDev &D, int nx, int ny, int nz,
                           const double *d_x, const double *d_y, const double *d_z,
                           double *d_v, float *d_v32, hipStream_t s)
{
    PC_REQUIRE(D.nsites <= kMaxSites, PISCES_ERR_UNSUPPORTED, "too many sites");
    const int K = pot_points((long long)nx * ny * nz);
    const long long threads = (long long)nx * ny * ((nz + K - 1) / K);
    const unsigned blocks = (unsigned)((threads + kPotThreads - 1) / kPotThreads);
    auto *kernel = K == 2 ? potential_grid_kernel<2> : potential_grid_kernel<1>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kPotThreads), 0, s, P, D, nx, ny, nz, d_x, d_y, d_z, d_v,
                       d_v32);
    PC_HIP(hipGetLastError());
}

void potential_grid_batched_launch(const PotParams &P, const PotTask *h_tasks, const PotTask *d_tasks,
                                   int ntasks, hipStream_t s)
{
    if (ntasks <= 0) return;
    long long points = 0, threads = 0;
    for (int i = 0; i < ntasks; ++i) points += (long long)h_tasks[i].nx * h_tasks[i].ny * h_tasks[i].nz;
    const int K = pot_points(points);
    for (int i = 0; i < ntasks; ++i) {
        const PotTask &t = h_tasks[i];
        threads = std::max(threads, (long long)t.nx * t.ny * ((t.nz + K - 1) / K));
    }
    const unsigned blocks = (unsigned)((threads + kPotThreads - 1) / kPotThreads);
    auto *kernel = K == 2 ? potential_grid_batched_kernel<2> : potential_grid_batched_kernel<1>;
    hipLaunchKernelGGL(kernel, dim3(blocks, ntasks), dim3(kPotThreads), 0, s, P, d_tasks);
    PC_HIP(hipGetLastError());
}

namespace {
// Dynamic LDS of a launch whose largest cluster has ns sites: all of it once
// the pairs of some cluster size up to that overflow the registers.
template <int NT> size_t scf_lds_bytes(int ns)
{
    static std::once_flag once;
    std::call_once(once, [] {
        for (const void *k : {reinterpret_cast<const void *>(water_scf_kernel<NT>),
                              reinterpret_cast<const void *>(water_scf_batched_kernel<NT>)})
            PC_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, Scf<NT>::LDS));
    });
    for (int m = 1; m <= ns; ++m)
        if (Scf<NT>::slots(m) > 0) return Scf<NT>::LDS;
    return (size_t)9 * ns * sizeof(double);
}
template <int NT> size_t scf_work_bytes(int ns)
{
    const int n = Scf<NT>::pairs(ns) - Scf<NT>::HELD - Scf<NT>::slots(ns);
    return n > 0 ? (size_t)n * Scf<NT>::SLOT_BYTES : 0;
}
}  // namespace

int water_scf_max_waters() { return kScfLarge / 3; }
int potential_max_sites() { return kMaxSites; }

size_t water_scf_work_bytes(int nw)
{
    return scf_threads(3 * nw) == kScfSmall ? scf_work_bytes<kScfSmall>(3 * nw) : scf_work_bytes<kScfLarge>(3 * nw);
}

// a launch per form that the batch holds, its LDS sized by the form's largest cluster
void water_scf_batched_launch(const ScfTask *h_tasks, const ScfTask *d_tasks, int ntasks, hipStream_t s)
{
    int small = 0, large = 0;  // sites of the largest cluster of each form
    for (int i = 0; i < ntasks; ++i) {
        const int ns = 3 * h_tasks[i].nw;
        int &m = scf_threads(ns) == kScfSmall ? small : large;
        m = std::max(m, ns);
    }
    if (small)
        hipLaunchKernelGGL((water_scf_batched_kernel<kScfSmall>), dim3(ntasks), dim3(kScfSmall),
                           scf_lds_bytes<kScfSmall>(small), s, d_tasks);
    if (large)
        hipLaunchKernelGGL((water_scf_batched_kernel<kScfLarge>), dim3(ntasks), dim3(kScfLarge),
                           scf_lds_bytes<kScfLarge>(large), s, d_tasks);
    PC_HIP(hipGetLastError());
}

void water_scf_launch(int nw, const double *d_sites, double *d_mu, double *d_epc, double *d_work,
                      int *d_info, hipStream_t s)
{
    PC_REQUIRE(nw > 0 && nw <= water_scf_max_waters(), PISCES_ERR_UNSUPPORTED,
               "too many waters for the dipole solve");
    const int ns = 3 * nw;
    if (scf_threads(ns) == kScfSmall)
        hipLaunchKernelGGL((water_scf_kernel<kScfSmall>), dim3(1), dim3(kScfSmall),
                           scf_lds_bytes<kScfSmall>(ns), s, nw, d_sites, d_mu, d_epc, d_work, d_info);
    else
        hipLaunchKernelGGL((water_scf_kernel<kScfLarge>), dim3(1), dim3(kScfLarge),
                           scf_lds_bytes<kScfLarge>(ns), s, nw, d_sites, d_mu, d_epc, d_work, d_info);
    PC_HIP(hipGetLastError());
}

}  // namespace pisces
