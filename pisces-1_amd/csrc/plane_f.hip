// plane_f.hip -- matrix-core plane kernels in FP64 and FP32 for gfx950: H*X
// (both precisions) and the kinetic preconditioner (FP64).
//
// The operators and their passes are those of plane.hip.  A workgroup stages
// one plane of one vector in LDS (rows c, columns i) and each of its waves
// owns one 16-row tile and NIT 16-column tiles of the plane: it loads, stages,
// accumulates and stores those elements, in the accumulator layout of the
// 16x16x4 matrix instructions (lane l, l16 = l % 16, lq = l / 16: A[l16][lq],
// B[lq][l16], D rows Acc<T>::row(lq, r) of column l16).
//
// What bounds these kernels is latency at the vector counts of a solve: a
// 64^3 pass is 64 planes per vector on 256 CUs.  So every operand a workgroup
// needs is requested before the first wait -- the plane, V or Y, the along-c
// matrix as held fragments of the wave's row tile (read from its transpose, 128
// contiguous bytes per row), the along-i matrix on its way to LDS -- and the
// column tiles of a row are split over CS waves, so that two waves per SIMD
// share the matrix cores (four splits: the same at 8 vectors, 1.14x slower at
// 32).  16-point tiles and k groups that lie entirely in the padding are
// skipped.  Measured, both passes (three for the preconditioner), us, before
// (matrix operands fetched inside the k loops, four waves) -> now:
//   64^3 x 8 vectors: H*X FP64 57.5 -> 39.1, FP32 38.6 -> 22.3, preconditioner
//   FP64 91.8 -> 62.5 (at x 1: 33.8 -> 18.7, 26.3 -> 13.4, 55.0 -> 29.8);
//   96^3 x 8: 304 -> 118, 143 -> 60, 509 -> 210.
// The matrix cores alone need 11.2 us for H*X FP64 at 64^3 x 8; the passes move
// 82 MB there (Y goes out and back between them).
#include "plane.hpp"

#include <mutex>

namespace pisces {

namespace {

template <typename T> __device__ inline const T *tmat(const AxisMats &m);
template <> __device__ inline const double *tmat<double>(const AxisMats &m) { return m.t64; }
template <> __device__ inline const float *tmat<float>(const AxisMats &m) { return m.t32; }

// Kernel shape for planes of at most 16 NT points per axis.
template <typename T, int NT> struct Cfg {
    // a 128-point FP64 plane leaves no LDS for the along-i matrix, and its
    // accumulators and fragments need the registers of two waves per SIMD
    static constexpr bool BIG = sizeof(T) == 8 && NT == 8;
    static constexpr int CS = BIG ? 1 : 2;          // column splits
    static constexpr int NIT = NT / CS;             // column tiles per wave
    static constexpr int THREADS = 64 * NT * CS;
    static constexpr int KF = 4 * NT;               // k-steps
    static constexpr int NP = 16 * NT;
    static constexpr int PAD = sizeof(T) == 8 ? 2 : 4;  // row padding in LDS
    static constexpr int VE = 16 / (int)sizeof(T);  // elements per 16-byte load
    static constexpr int TV = BIG ? 1 : (NP * NP / VE + THREADS - 1) / THREADS;
    static constexpr size_t plane_bytes = (size_t)NP * (NP + PAD) * sizeof(T);
};

template <typename T> struct Vec16;
template <> struct Vec16<double> { typedef f64x2 type; };
template <> struct Vec16<float> { typedef f32x4 type; };

// element `off` (in elements, 32-bit) of a wave-uniform base
template <typename T> __device__ __forceinline__ T at(gptr<const T> base, unsigned off)
{
    return *reinterpret_cast<gptr<const T>>(reinterpret_cast<gptr<const char>>(base) +
                                            off * (unsigned)sizeof(T));
}

// The wave's place in the plane and its elements' offsets.
template <typename T, int NT> struct Own {
    typedef Cfg<T, NT> C;
    int tc, v0, l16, lq, ntc, nti;
    bool active;
    __device__ __forceinline__ explicit Own(const Geo &g)
    {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        l16 = lane & 15;
        lq = lane >> 4;
        tc = wave % NT;
        v0 = (wave / NT) * C::NIT;
        ntc = (g.nc + 15) / 16;
        nti = (g.ni + 15) / 16;
        active = tc < ntc && v0 < nti;
    }
    __device__ __forceinline__ int row(int r) const { return 16 * tc + Acc<T>::row(lq, r); }
    __device__ __forceinline__ int col(int v) const { return 16 * (v0 + v) + l16; }
};

// Owned elements, zero outside the plane; every lane loads unconditionally
// (out-of-plane elements from (0, 0)) so that the loads issue back to back.
template <typename T, int NT>
__device__ __forceinline__ void own_load(const T *src, long long base, const Geo &g,
                                         const Own<T, NT> &o, T (&x)[Cfg<T, NT>::NIT][4])
{
    const gptr<const T> s = glb(src) + base;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = o.row(r);
        const unsigned oc = (unsigned)c * (unsigned)g.cs;
#pragma unroll
        for (int v = 0; v < Cfg<T, NT>::NIT; ++v) {
            const int i = o.col(v);
            const bool ok = c < g.nc && i < g.ni;
            const T y = at<T>(s, ok ? oc + (unsigned)i : 0u);
            x[v][r] = ok ? y : T(0);
        }
    }
}

template <typename T, int NT>
__device__ __forceinline__ void own_put(T *P, int pitch, const Own<T, NT> &o,
                                        const T (&x)[Cfg<T, NT>::NIT][4])
{
#pragma unroll
    for (int v = 0; v < Cfg<T, NT>::NIT; ++v)
        if (o.v0 + v < o.nti)
#pragma unroll
            for (int r = 0; r < 4; ++r) P[o.row(r) * pitch + o.col(v)] = x[v][r];
}

// A fragments of matrix M for the wave's row tile, from its transpose Mt
// (row-major, np x np): af[s] = M[16 tc + l16][4 s + lq] = Mt[4 s + lq][16 tc + l16]
template <typename T, int NT>
__device__ __forceinline__ void a_frag(const T *Mt, int np, const Own<T, NT> &o, T (&af)[4 * NT])
{
    const gptr<const T> m = glb(Mt);
    const unsigned c = 16 * o.tc + o.l16;
#pragma unroll
    for (int s = 0; s < 4 * NT; ++s) {
        const int k = 4 * s + o.lq;
        af[s] = at<T>(m, k < np && (int)c < np ? (unsigned)(k * np) + c : 0u);
    }
}

// A row-major np x np matrix on its way to LDS (pitch np + PAD): mat_load
// requests the thread's 16-byte pieces, mat_put stores them.
template <typename T, int NT> struct MatStage {
    typedef Cfg<T, NT> C;
    typedef typename Vec16<T>::type V;
    V v[C::TV];
    __device__ __forceinline__ void load(const T *M, int np)
    {
        const gptr<const V> m = reinterpret_cast<gptr<const V>>(glb(M));
        const int n = np * np / C::VE;
#pragma unroll
        for (int u = 0; u < C::TV; ++u) {
            const int e = threadIdx.x + u * C::THREADS;
            v[u] = at<V>(m, e < n ? e : 0);
        }
    }
    __device__ __forceinline__ void put(T *L, int np) const
    {
        const int n = np * np / C::VE, q = np / C::VE;
#pragma unroll
        for (int u = 0; u < C::TV; ++u) {
            const int e = threadIdx.x + u * C::THREADS;
            const int k = e / q, i = e - k * q;
            if (e < n) *reinterpret_cast<V *>(L + k * (np + C::PAD) + i * C::VE) = v[u];
        }
    }
};

// acc(c, i) += sum_k M[c][k] P[k][i] over the rows k of the plane
template <typename T, int NT>
__device__ __forceinline__ void mul_c(const T (&af)[4 * NT], const T *P, int pitch, const Own<T, NT> &o,
                                      typename Acc<T>::type (&acc)[Cfg<T, NT>::NIT])
{
    const T *b = P + o.lq * pitch + 16 * o.v0 + o.l16;
#pragma unroll
    for (int s4 = 0; s4 < NT; ++s4) {
        if (s4 >= o.ntc) break;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int v = 0; v < Cfg<T, NT>::NIT; ++v)
                acc[v] = mma(af[4 * s4 + q], b[(16 * s4 + 4 * q) * pitch + 16 * v], acc[v]);
    }
}

// acc(c, i) += sum_k P[c][k] M[k][i] over the columns k of the plane; M in LDS
// (Ml, pitch as the plane) or, for the largest planes, in global memory
template <typename T, int NT>
__device__ __forceinline__ void mul_i(const T *P, int pitch, const T *Ml, const T *M, int np,
                                      const Own<T, NT> &o,
                                      typename Acc<T>::type (&acc)[Cfg<T, NT>::NIT])
{
    const T *a = P + (16 * o.tc + o.l16) * pitch + o.lq;
    const T *b = Ml + o.lq * pitch + 16 * o.v0 + o.l16;
    const gptr<const T> g = glb(M);
#pragma unroll
    for (int s4 = 0; s4 < NT; ++s4) {
        if (s4 >= o.nti) break;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = 16 * s4 + 4 * q;
            const T av = a[k];
#pragma unroll
            for (int v = 0; v < Cfg<T, NT>::NIT; ++v) {
                const T bv = Cfg<T, NT>::BIG
                                 ? (o.v0 + v < o.nti ? at<T>(g, (unsigned)((k + o.lq) * np + o.col(v))) : T(0))
                                 : b[k * pitch + 16 * v];
                acc[v] = mma(av, bv, acc[v]);
            }
        }
    }
}

// ------------------------------------------------------------------ H*X
// Plane p of one pass of job J: pass A (plane (i,j) at k) Y = V o X + Ty X
// along j, pass B (plane (i,k) at j) Y += Tz X along k + X Tx along i.  The
// kinetic matrices are symmetric, so they are their own transposes.
template <typename T, int PASS, int NT>
__device__ __forceinline__ void hx_plane(const HxJob &J, int p, unsigned char *smem)
{
    typedef Cfg<T, NT> C;
    typedef typename Acc<T>::type acc_t;
    const AxisMats &Mi = J.ax[0];
    const AxisMats &Mc = J.ax[PASS == 0 ? 1 : 2];
    Geo g;
    if (!geo_of(PASS, J.nx, J.ny, J.nz, J.nvec, J.ld, Mi.np, Mc.np, p, g)) return;
    const Own<T, NT> o(g);
    const int pitch = g.npi + C::PAD;
    T *P = reinterpret_cast<T *>(smem);
    T *Ml = P + g.npc * pitch;
    const T *X = static_cast<const T *>(J.X);
    T *Y = static_cast<T *>(J.Y);
    const T *W = PASS == 0 ? static_cast<const T *>(J.V) : Y;  // V (pass A) or Y (pass B)
    T af[C::KF], xb[C::NIT][4], wb[C::NIT][4];
    MatStage<T, NT> ti;
    if (o.active) own_load<T, NT>(X, g.base, g, o, xb);
    if (PASS == 1 && !C::BIG) ti.load(tmat<T>(Mi), g.npi);
    if (o.active) {
        a_frag<T, NT>(tmat<T>(Mc), g.npc, o, af);
        own_load<T, NT>(W, PASS == 0 ? g.vbase : g.base, g, o, wb);
        own_put<T, NT>(P, pitch, o, xb);
    }
    if (PASS == 1 && !C::BIG) ti.put(Ml, g.npi);
    __syncthreads();
    if (!o.active) return;
    acc_t acc[C::NIT];
    // FP64 pass A accumulates onto V o X; the others add their sum at the end
    constexpr bool INIT = PASS == 0 && sizeof(T) == 8;
#pragma unroll
    for (int v = 0; v < C::NIT; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (PASS == 0) wb[v][r] *= xb[v][r];
            acc[v][r] = INIT ? wb[v][r] : T(0);
        }
    mul_c<T, NT>(af, P, pitch, o, acc);
    if (PASS == 1) mul_i<T, NT>(P, pitch, Ml, tmat<T>(Mi), g.npi, o, acc);
    const gptr<T> y = glb(Y) + g.base;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = o.row(r);
        const unsigned oc = (unsigned)c * (unsigned)g.cs;
#pragma unroll
        for (int v = 0; v < C::NIT; ++v) {
            const int i = o.col(v);
            if (c < g.nc && i < g.ni)
                *reinterpret_cast<gptr<T>>(reinterpret_cast<gptr<char>>(y) +
                                           (oc + (unsigned)i) * (unsigned)sizeof(T)) =
                    INIT ? acc[v][r] : wb[v][r] + acc[v][r];
        }
    }
}

template <typename T, int PASS, int NT>
__global__ void __launch_bounds__((Cfg<T, NT>::THREADS)) hx_f_kernel(const HxJob *__restrict__ jobs)
{
    extern __shared__ __align__(16) unsigned char smem[];
    hx_plane<T, PASS, NT>(jobs[plane_y(PASS == 1)], plane_x(PASS == 1), smem);
}

template <typename T, int PASS, int NT>
__global__ void __launch_bounds__((Cfg<T, NT>::THREADS)) hx_f_one_kernel(HxJob J)
{
    extern __shared__ __align__(16) unsigned char smem[];
    hx_plane<T, PASS, NT>(J, plane_x(PASS == 1), smem);
}

// ------------------------------------------------------------------ H*X, small grids
// Both passes in one launch for grids of at most 32 points per axis: a workgroup
// owns one 16 x 16 tile of the (i,j) plane at k, contracts the plane along j and
// i on the matrix cores as above, and adds the z sum of its points on the VALU,
//   Y(i,j,k) += sum_k' Tz[k][k'] X(i,j,k'),
// reading the other planes' tiles straight from the caches (a vector is at most
// 256 KB).  There is no intermediate Y and no second launch.  The four waves split
// k' and the two contractions; their sums meet in LDS in a fixed order.
constexpr int kSmallN = 32, kSmallThreads = 256;

template <typename T>
__global__ void __launch_bounds__(kSmallThreads) hx_small_kernel(HxJob J, int nti, int ntiles)
{
    typedef typename Acc<T>::type acc_t;
    constexpr int PITCH = kSmallN + (sizeof(T) == 8 ? 2 : 4), KZ = kSmallN / 4;
    __shared__ T P[kSmallN * PITCH], Ml[kSmallN * PITCH];
    __shared__ T red[3][4][64];  // wave - 1, element, lane
    const int pv = blockIdx.x / ntiles, tile = blockIdx.x - pv * ntiles;
    const int v = pv / J.nz, k = pv - v * J.nz;
    const int lane = threadIdx.x & 63, zq = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int r0 = 16 * (tile / nti), i = 16 * (tile % nti) + l16;
    const int nx = J.nx, ny = J.ny, nz = J.nz;
    const unsigned plane = (unsigned)nx * ny;
    const gptr<const T> X = glb(static_cast<const T *>(J.X)) + J.ld * v;
    const gptr<const T> xp = X + (size_t)k * plane;
    // the lane's four points of the tile
    unsigned off[4];
    bool ok[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = r0 + Acc<T>::row(lq, r);
        ok[r] = c < ny && i < nx;
        off[r] = ok[r] ? (unsigned)(c * nx + i) : 0u;
    }
    // the plane and Tx on their way to LDS, this wave's planes k', V, Ty
    T ps[4], ms[4], xz[KZ][4], tz[KZ], xk[4], vk[4], af[8];
    const int pi = threadIdx.x & 31, pc = threadIdx.x >> 5;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int c = pc + 8 * u;
        const bool in = pi < nx && c < ny;
        ps[u] = at<T>(xp, in ? (unsigned)(c * nx + pi) : 0u);
        ps[u] = in ? ps[u] : T(0);
        ms[u] = glb(tmat<T>(J.ax[0]))[c * kSmallN + pi];
    }
    const gptr<const T> Tz = glb(tmat<T>(J.ax[2])) + k * kSmallN;
    const int zs = (nz + 3) / 4, k0 = zs * zq;
#pragma unroll
    for (int u = 0; u < KZ; ++u) {
        const bool on = u < zs && k0 + u < nz;
        tz[u] = T(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) xz[u][r] = T(0);
        if (on) {
            tz[u] = Tz[k0 + u];
            const gptr<const T> xq = X + (size_t)(k0 + u) * plane;
#pragma unroll
            for (int r = 0; r < 4; ++r) xz[u][r] = at<T>(xq, off[r]);
        }
    }
    if (zq == 0) {
        const gptr<const T> V = glb(static_cast<const T *>(J.V)) + (size_t)k * plane;
        const gptr<const T> Ty = glb(tmat<T>(J.ax[1]));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            xk[r] = at<T>(xp, off[r]);
            vk[r] = at<T>(V, off[r]);
        }
#pragma unroll
        for (int s = 0; s < 8; ++s) af[s] = Ty[(4 * s + lq) * kSmallN + r0 + l16];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        P[(pc + 8 * u) * PITCH + pi] = ps[u];
        Ml[(pc + 8 * u) * PITCH + pi] = ms[u];
    }
    __syncthreads();
    acc_t acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = zq == 0 && ok[r] ? vk[r] * xk[r] : T(0);
    const int sy = (ny + 3) / 4, sx = (nx + 3) / 4;  // k-steps that hold points
    if (zq == 0) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (s < sy) acc = mma(af[s], P[(4 * s + lq) * PITCH + i], acc);
    } else if (zq == 1) {
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (s < sx) acc = mma(P[(r0 + l16) * PITCH + 4 * s + lq], Ml[(4 * s + lq) * PITCH + i], acc);
    }
    T z[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int u = 0; u < KZ; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) z[r] += tz[u] * xz[u][r];
#pragma unroll
    for (int r = 0; r < 4; ++r) z[r] += acc[r];
    if (zq > 0)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[zq - 1][r][lane] = z[r];
    __syncthreads();
    if (zq > 0) return;
    const gptr<T> y = glb(static_cast<T *>(J.Y)) + (J.ld * v + (long long)k * plane);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const T s = z[r] + ((red[0][r][lane] + red[1][r][lane]) + red[2][r][lane]);
        if (ok[r]) y[off[r]] = s;
    }
}

// ------------------------------------------------------------------ preconditioner
// Passes as in plane.hip; passes 1 and 2 work in place in dst, where every
// plane is read (into LDS) and written by its one workgroup only.
template <int PASS, int NT>
__device__ __forceinline__ void fdm_plane(const FdmTask &t, int p, unsigned char *smem)
{
    typedef double T;
    typedef Cfg<T, NT> C;
    const AxisMats &Mx = t.ax[0], &My = t.ax[1], &Mz = t.ax[2];
    const AxisMats &Mc = PASS == 1 ? Mz : My;
    Geo g;
    if (!geo_of(PASS == 1 ? 1 : 0, Mx.n, My.n, Mz.n, 1, 0, Mx.np, Mc.np, p, g)) return;
    const Own<T, NT> o(g);
    const int pitch = g.npi + C::PAD;
    T *P = reinterpret_cast<T *>(smem);
    T *Ml = P + g.npc * pitch;
    // along c: Qy^T (pass 0), Qz^T then Qz (pass 1), Qy (pass 2), each read
    // from its transpose; along i: Qx (pass 0), Qx^T (pass 2)
    const T *Mi = PASS == 0 ? Mx.q64 : Mx.qt64;
    T af[C::KF], a2[C::KF], xb[C::NIT][4];
    MatStage<T, NT> mi;
    T lx[C::NIT], lz[4], ly = 0.0;
    if (o.active) own_load<T, NT>(static_cast<const T *>(PASS == 0 ? t.src : t.dst), g.base, g, o, xb);
    if (PASS != 1 && !C::BIG) mi.load(Mi, g.npi);
    if (o.active) {
        a_frag<T, NT>(PASS == 2 ? My.qt64 : Mc.q64, g.npc, o, af);
        if (PASS == 1) {
            if (!C::BIG) a_frag<T, NT>(Mz.qt64, g.npc, o, a2);
#pragma unroll
            for (int v = 0; v < C::NIT; ++v) lx[v] = at<T>(glb(Mx.lam), o.col(v) < g.ni ? o.col(v) : 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) lz[r] = at<T>(glb(Mz.lam), o.row(r) < g.nc ? o.row(r) : 0);
            ly = glb(My.lam)[g.pl];
        }
        own_put<T, NT>(P, pitch, o, xb);
    }
    if (PASS != 1 && !C::BIG) mi.put(Ml, g.npi);
    __syncthreads();
    f64x4 acc[C::NIT];
#pragma unroll
    for (int v = 0; v < C::NIT; ++v) acc[v] = f64x4{0.0, 0.0, 0.0, 0.0};
    if (o.active) {
        if (PASS == 0) mul_i<T, NT>(P, pitch, Ml, Mi, g.npi, o, acc);  // P Qx
        else mul_c<T, NT>(af, P, pitch, o, acc);                       // Qz^T P, Qy P
        if (PASS == 1 && C::BIG) a_frag<T, NT>(Mz.qt64, g.npc, o, a2);
    }
    __syncthreads();  // every wave has read the plane
    if (o.active) {
#pragma unroll
        for (int v = 0; v < C::NIT; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                T x = acc[v][r];
                if (PASS == 1) {
                    // plane (i = a, c = z index) at fixed j = b
                    T den = 1.0;
                    if (o.col(v) < g.ni && o.row(r) < g.nc) {
                        den = lx[v] + ly + lz[r] - t.shift;
                        if (t.absden) den = fabs(den);
                        if (fabs(den) < t.floor) den = den < 0 ? -t.floor : t.floor;
                    }
                    x *= t.scale / den;
                }
                xb[v][r] = x;
                acc[v][r] = 0.0;
            }
        own_put<T, NT>(P, pitch, o, xb);
    }
    __syncthreads();
    if (!o.active) return;
    if (PASS == 0) mul_c<T, NT>(af, P, pitch, o, acc);                      // Qy^T (.)
    else if (PASS == 1) mul_c<T, NT>(a2, P, pitch, o, acc);                 // Qz (.)
    else mul_i<T, NT>(P, pitch, Ml, Mi, g.npi, o, acc);                     // (.) Qx^T
    const gptr<T> d = glb(static_cast<T *>(t.dst)) + g.base;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = o.row(r);
#pragma unroll
        for (int v = 0; v < C::NIT; ++v)
            if (c < g.nc && o.col(v) < g.ni)
                *reinterpret_cast<gptr<T>>(reinterpret_cast<gptr<char>>(d) +
                                           ((unsigned)c * (unsigned)g.cs + o.col(v)) * 8u) = acc[v][r];
    }
}

template <int PASS, int NT>
__global__ void __launch_bounds__((Cfg<double, NT>::THREADS)) fdm_f64_kernel(const FdmTask *__restrict__ tasks)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fdm_plane<PASS, NT>(tasks[plane_y(PASS == 1)], plane_x(PASS == 1), smem);
}

template <int PASS, int NT>
__global__ void __launch_bounds__((Cfg<double, NT>::THREADS)) fdm_f64_one_kernel(FdmOne one)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fdm_plane<PASS, NT>(task_of(one, plane_y(PASS == 1), 8, 8), plane_x(PASS == 1), smem);
}

// ------------------------------------------------------------------ launches
template <typename T, int NT>
void hx_nt_launch(const HxJob *d, const HxJob *one, int n, int pa, int pb, hipStream_t s)
{
    typedef Cfg<T, NT> C;
    static std::once_flag once;
    std::call_once(once, [] {
        allow_lds(hx_f_kernel<T, 0, NT>);
        allow_lds(hx_f_kernel<T, 1, NT>);
        allow_lds(hx_f_one_kernel<T, 0, NT>);
        allow_lds(hx_f_one_kernel<T, 1, NT>);
    });
    const size_t la = C::plane_bytes, lb = C::BIG ? la : 2 * la;
    if (one) {
        hipLaunchKernelGGL((hx_f_one_kernel<T, 0, NT>), dim3(pa), dim3(C::THREADS), la, s, *one);
        hipLaunchKernelGGL((hx_f_one_kernel<T, 1, NT>), dim3(pb), dim3(C::THREADS), lb, s, *one);
        return;
    }
    hipLaunchKernelGGL((hx_f_kernel<T, 0, NT>), dim3(pa, n), dim3(C::THREADS), la, s, d);
    hipLaunchKernelGGL((hx_f_kernel<T, 1, NT>), dim3(pb, n), dim3(C::THREADS), lb, s, d);
}

// Most tiles (workgroups) for which the one-launch form is taken: beyond about
// four a CU its repeated reads of the vector cost more than the second launch.
// us, one launch / two: 12^3 x 1 3.5 / 6.5 (FP64), 32^3 x 1 4.1 / 7.7, x 4 5.6 / 8.0,
// x 8 (1024 tiles) 8.6 / 8.5, x 16 14.0 / 10.8; FP32 32^3 x 1 3.6 / 6.7, x 8 5.7 / 7.1,
// x 16 9.7 / 8.1.
constexpr int kSmallTiles = 1000;

template <typename T>
void hx_t_launch(const HxJob *d, const HxJob *one, int n, int pa, int pb, int np, hipStream_t s)
{
    const int nti = one ? (one->nx + 15) / 16 : 0, ntiles = one ? nti * ((one->ny + 15) / 16) : 0;
    if (one && np <= 32 && (long long)pa * ntiles <= kSmallTiles)
        hipLaunchKernelGGL((hx_small_kernel<T>), dim3(pa * ntiles), dim3(kSmallThreads), 0, s, *one, nti, ntiles);
    else if (np <= 32) hx_nt_launch<T, 2>(d, one, n, pa, pb, s);
    else if (np <= 64) hx_nt_launch<T, 4>(d, one, n, pa, pb, s);
    else if (np <= 96) hx_nt_launch<T, 6>(d, one, n, pa, pb, s);
    else hx_nt_launch<T, 8>(d, one, n, pa, pb, s);
}

template <int NT>
void fdm_nt_launch(const FdmTask *d, const FdmOne *one, int n, int planes, hipStream_t s)
{
    typedef Cfg<double, NT> C;
    static std::once_flag once;
    std::call_once(once, [] {
        allow_lds(fdm_f64_kernel<0, NT>);
        allow_lds(fdm_f64_kernel<1, NT>);
        allow_lds(fdm_f64_kernel<2, NT>);
        allow_lds(fdm_f64_one_kernel<0, NT>);
        allow_lds(fdm_f64_one_kernel<1, NT>);
        allow_lds(fdm_f64_one_kernel<2, NT>);
    });
    const size_t l1 = C::plane_bytes, l2 = C::BIG ? l1 : 2 * l1;
    const dim3 grid(planes, n), blk(C::THREADS);
    if (one) {
        hipLaunchKernelGGL((fdm_f64_one_kernel<0, NT>), grid, blk, l2, s, *one);
        hipLaunchKernelGGL((fdm_f64_one_kernel<1, NT>), grid, blk, l1, s, *one);
        hipLaunchKernelGGL((fdm_f64_one_kernel<2, NT>), grid, blk, l2, s, *one);
        return;
    }
    hipLaunchKernelGGL((fdm_f64_kernel<0, NT>), grid, blk, l2, s, d);
    hipLaunchKernelGGL((fdm_f64_kernel<1, NT>), grid, blk, l1, s, d);
    hipLaunchKernelGGL((fdm_f64_kernel<2, NT>), grid, blk, l2, s, d);
}

}  // namespace

void hx_f_launch(const HxJob *d_jobs, const HxJob *one, int njobs, int max_planes_a, int max_planes_b, int max_n,
                 int precision, hipStream_t s)
{
    const int np = axis_pad(max_n);
    if (precision == PISCES_FP32) hx_t_launch<float>(d_jobs, one, njobs, max_planes_a, max_planes_b, np, s);
    else hx_t_launch<double>(d_jobs, one, njobs, max_planes_a, max_planes_b, np, s);
    PC_HIP(hipGetLastError());
}

void fdm_f64_launch(const FdmTask *d_tasks, const FdmOne *one, int ntasks, int max_n, hipStream_t s)
{
    const int np = axis_pad(max_n);
    // planes per pass: the largest of ny (pass 1) and nz (passes 0, 2) <= max_n
    if (np <= 32) fdm_nt_launch<2>(d_tasks, one, ntasks, max_n, s);
    else if (np <= 64) fdm_nt_launch<4>(d_tasks, one, ntasks, max_n, s);
    else if (np <= 96) fdm_nt_launch<6>(d_tasks, one, ntasks, max_n, s);
    else fdm_nt_launch<8>(d_tasks, one, ntasks, max_n, s);
    PC_HIP(hipGetLastError());
}

}  // namespace pisces
