// plane.hip -- matrix-core plane kernels for gfx950: the split-BF16 forms of H*X
// and of the kinetic fast-diagonalisation preconditioner, and the dispatch to
// the FP64 and FP32 forms (plane_f.hip).
//
// Both operators are sums or products of dense 1-D matrices applied along the
// axes of the x-fastest grid (g = i + nx*(j + ny*k)).  A workgroup stages one
// 2-D plane of one vector in LDS -- rows c, columns i, both padded to multiples of
// 32 -- and contracts it along one or both of its axes:
//   along c:  D(c, i) += sum_k Mc[c][k] P[k][i]   (A = Mc from HBM/L2, B = plane)
//   along i:  D(c, i) += sum_k P[c][k] Mi[k][i]   (A = plane, B = Mi)
// on 16 x 16 output tiles.  For planes of at most 16 NT points an axis it has NT CS
// waves: each takes one tile row and, of its columns, one of CS equal parts, two
// column tiles at a time in the contraction along c (two accumulator chains).
//
// Instruction operand layouts (lane l, l16 = l % 16, lq = l / 16):
//   f64 16x16x4 : A[l16][lq], B[lq][l16], D element r = D[lq + 4r][l16]
//   f32 16x16x4 : A[l16][lq], B[lq][l16], D element r = D[4lq + r][l16]
//   bf16 16x16x32 (f32 acc): A[l16][8lq + e], B[8lq + e][l16], e < 8,
//                 D element r = D[4lq + r][l16]
// The split-BF16 form stores every operand as hi = bf16(x), lo = bf16(x - hi)
// and accumulates hi*hi + hi*lo + lo*hi in FP32 (about 16 significant bits).
// Its B operand needs 8 consecutive k per lane, so the plane is kept in LDS
// transposed (i-major) for contractions along c and as is (c-major) for
// contractions along i, and the matrix Mi is read as Mi^T (row-major); every
// operand fetch is then one 16-byte load.
//
// H*X: pass A, plane (i,j) at k:  Y  = V o X + Ty along j
//      pass B, plane (i,k) at j:  Y += Tx along i + Tz along k
// Preconditioner t = scale (T - shift)^{-1} r through the eigenbases
// (T_a = Q_a diag(lam_a) Q_a^T), three passes:
//      0, plane (i,j) at k:  W = Qy^T (P Qx)                    (r -> W)
//      1, plane (i,k) at j:  W = Qz (S o (Qz^T P)),  S = scale / (lam_x + lam_y + lam_z - shift)
//      2, plane (i,j) at k:  t = (Qy P) Qx^T                     (W -> t)
// with |lam_x + lam_y + lam_z - shift| floored at `floor`.
#include "plane.hpp"

#include <algorithm>
#include <cstdlib>
#include <mutex>

namespace pisces {

namespace {

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ uint16_t bf16_rne(float x)
{
    unsigned int u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
// (x0, x1) as packed BF16 pairs hi = bf16(x), lo = bf16(x - hi), rounded to
// nearest even by the hardware conversion
__device__ __forceinline__ unsigned pack_bf16(float x0, float x1)
{
    const f32x2 x = {x0, x1};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2));
}
__device__ __forceinline__ void split2(float x0, float x1, unsigned &h, unsigned &l)
{
    h = pack_bf16(x0, x1);
    l = pack_bf16(x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xffff0000u));
}
__device__ __forceinline__ bf16x8 ld8(const uint16_t *p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p));
}
__device__ __forceinline__ bf16x8 ld8(gptr<const uint16_t> p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<gptr<const u32x4>>(p));
}
__device__ __forceinline__ f32x4 mma_bf(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ------------------------------------------------------------------ owned tiles
// A workgroup holds one plane.  Its NT x CS waves split the plane's 16 x 16
// tiles: wave (tc, h) owns row tile tc and the NIT column tiles from h NIT on;
// in each, lane (l16, lq) holds rows 4 lq + r (r < 4) of column l16 -- the
// accumulator layout of the f32-accumulating MFMAs.  Global loads, LDS staging
// and global stores follow this ownership, so a wave combines its results with
// values it loaded itself, and a plane's rows move HBM -> registers -> LDS
// without a layout change.  Everything a wave needs from memory is requested
// before the first wait: at the vector counts of a solve these kernels are
// bound by the latency of that chain, not by HBM, LDS or the matrix cores.
// Measured, all passes, us, before (four waves a plane, two row tiles each above
// 64 points, four planes per preconditioner workgroup at 64) -> now:
//   H*X 96^3 x 8 70.4 -> 50.0, 128^3 x 8 228 -> 143, 48^3 x 128 98 -> 75,
//   64^3 x 32 48.6 -> 47.8; preconditioner 64^3 x 1 50.4 -> 18.1, x 32 70.4 ->
//   61.5, x 128 209 -> 186, 96^3 x 8 104 -> 73.
// At 64^3 x 128 H*X moves 5.2 MB a vector between its passes and HBM at 4.6
// TB/s, near the rate of a plain copy.
template <int NT, int CS> struct Cfg {
    static constexpr int NIT = NT / CS;     // column tiles per wave
    static constexpr int THREADS = 64 * NT * CS;
    static constexpr int KS = NT / 2;       // k-steps of the bf16 MFMA
    // the along-i matrix as held fragments of the wave's columns, requested with
    // the plane; for larger planes they do not fit the registers and are read
    // where they are used
    static constexpr bool HOLD = NT <= 4 && CS == 2;
};

template <int NT, int CS> struct Own {
    static constexpr int NIT = Cfg<NT, CS>::NIT;
    int tc, v0, l16, lq, ntc, nti, npc, npi;
    bool active;  // some of the wave's tiles hold points of the plane
    __device__ __forceinline__ explicit Own(const Geo &g)
    {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        l16 = lane & 15;
        lq = lane >> 4;
        tc = wave % NT;
        v0 = (wave / NT) * NIT;
        ntc = (g.nc + 15) / 16;
        nti = (g.ni + 15) / 16;
        npc = g.npc / 16;  // staged tiles: the matrix instruction reads 32 k at a time
        npi = g.npi / 16;
        active = tc < ntc && v0 < nti;
    }
    __device__ __forceinline__ int row(int r) const { return 16 * tc + 4 * lq + r; }
    __device__ __forceinline__ int col(int v) const { return 16 * (v0 + v) + l16; }
};

// element `off` (in elements, 32-bit) of a wave-uniform base
template <typename T> __device__ __forceinline__ T at(gptr<const T> base, unsigned off)
{
    return *reinterpret_cast<gptr<const T>>(reinterpret_cast<gptr<const char>>(base) +
                                            off * (unsigned)sizeof(T));
}

// Owned plane values as FP32 (zero outside the n_c x n_i plane) from FP64,
// FP32 or BF16 (uint16_t bit patterns) storage.  Every lane loads
// unconditionally -- out-of-plane elements from the plane's (0, 0) -- so the
// loads issue back to back, and the value is selected afterwards.
template <typename S> __device__ __forceinline__ float as_f32(S v) { return (float)v; }
template <> __device__ __forceinline__ float as_f32<uint16_t>(uint16_t v)
{
    return __uint_as_float((unsigned int)v << 16);
}
template <typename S, int NT, int CS>
__device__ __forceinline__ void own_load(const S *src, long long base, const Geo &g, const Own<NT, CS> &o,
                                         float (&x)[Own<NT, CS>::NIT][4])
{
    const gptr<const S> s = glb(src) + base;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = o.row(r);
        const unsigned oc = (unsigned)c * (unsigned)g.cs;
#pragma unroll
        for (int v = 0; v < Own<NT, CS>::NIT; ++v) {
            const int i = o.col(v);
            const bool ok = c < g.nc && i < g.ni;
            const float y = as_f32(at<S>(s, ok ? oc + (unsigned)i : 0u));
            x[v][r] = ok ? y : 0.f;
        }
    }
}

// Row padding (BF16 elements) of the split planes in LDS: a row of a 64-point
// plane spans 64 + kBf2Pad elements (16 and 24 measured no faster)
constexpr int kBf2Pad = 8;

// Exchange a dword with the neighbouring lane (DPP quad_perm 1,0,3,2).
__device__ __forceinline__ unsigned swap_adj(unsigned x)
{
    return (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);
}

// Split one owned tile column (rows cb .. cb+3 of column i) into the LDS
// plane: i-major (Pt, pitch pt) and/or c-major (Pc, pitch pc); a null pointer
// skips a layout.  For the c-major rows the lanes of a column pair (i even,
// i + 1) meet in one dword: the even lane writes rows cb, cb+1, the odd lane
// rows cb+2, cb+3.  Every lane of the wave must take part.
__device__ __forceinline__ void put_tile(const float (&x)[4], int cb, int i, int pt, int pc,
                                         uint16_t *Pth, uint16_t *Ptl, uint16_t *Pch, uint16_t *Pcl)
{
    unsigned h01, h23, l01, l23;
    split2(x[0], x[1], h01, l01);
    split2(x[2], x[3], h23, l23);
    if (Pth) {
        u32x2 vh, vl;
        vh[0] = h01; vh[1] = h23;
        vl[0] = l01; vl[1] = l23;
        *reinterpret_cast<u32x2 *>(Pth + i * pt + cb) = vh;
        *reinterpret_cast<u32x2 *>(Ptl + i * pt + cb) = vl;
    }
    if (Pch) {
        const bool odd = i & 1;
        const unsigned hr = swap_adj(odd ? h01 : h23), lr = swap_adj(odd ? l01 : l23);
        const unsigned hm = odd ? h23 : h01, lm = odd ? l23 : l01;
        const unsigned hlo = odd ? hr : hm, hhi = odd ? hm : hr;  // columns i & ~1, i | 1
        const unsigned llo = odd ? lr : lm, lhi = odd ? lm : lr;
        const int row = cb + (odd ? 2 : 0), col = i & ~1;
        *reinterpret_cast<unsigned *>(Pch + row * pc + col) = (hlo & 0xffffu) | (hhi << 16);
        *reinterpret_cast<unsigned *>(Pch + (row + 1) * pc + col) = (hlo >> 16) | (hhi & 0xffff0000u);
        *reinterpret_cast<unsigned *>(Pcl + row * pc + col) = (llo & 0xffffu) | (lhi << 16);
        *reinterpret_cast<unsigned *>(Pcl + (row + 1) * pc + col) = (llo >> 16) | (lhi & 0xffff0000u);
    }
}

// The owned tiles into LDS, zeros of the padding included (the contractions
// read whole 32-point k-steps).
template <int NT, int CS>
__device__ __forceinline__ void own_put(const float (&x)[Own<NT, CS>::NIT][4], const Geo &g, const Own<NT, CS> &o,
                                        uint16_t *Pth, uint16_t *Ptl, uint16_t *Pch, uint16_t *Pcl)
{
    if (o.tc >= o.npc) return;
#pragma unroll
    for (int v = 0; v < Own<NT, CS>::NIT; ++v)
        if (o.v0 + v < o.npi)
            put_tile(x[v], 16 * o.tc + 4 * o.lq, o.col(v), g.npc + kBf2Pad, g.npi + kBf2Pad, Pth, Ptl,
                     Pch, Pcl);
}

// Fragments of a row-major split matrix (leading dimension np): rows
// 16 t + l16, columns 32 s + 8 lq .. + 7 -- the A operand of row tile t, or the
// B operand of column tile t of its transpose.
template <int KS> struct Frag {
    bf16x8 h[KS], l[KS];
    template <typename P> __device__ __forceinline__ void load(P Mh, P Ml, int ld, int t, int l16, int lq, int ks)
    {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int e = s < ks ? (16 * t + l16) * ld + 32 * s + 8 * lq : 0;
            h[s] = ld8(Mh + e);
            l[s] = ld8(Ml + e);
        }
    }
};

// acc += A B over ks k-steps, split-BF16: hi*hi + hi*lo + lo*hi
template <int KS>
__device__ __forceinline__ void mm(const Frag<KS> &a, const Frag<KS> &b, int ks, f32x4 &acc)
{
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if (s >= ks) break;
        acc = mma_bf(a.h[s], b.h[s], acc);
        acc = mma_bf(a.h[s], b.l[s], acc);
        acc = mma_bf(a.l[s], b.h[s], acc);
    }
}

// acc(c, i) += sum_k M[c][k] P[k][i]: A = held fragments of the wave's row
// tile of M, B = the i-major plane
template <int NT, int CS>
__device__ __forceinline__ void mul_c(const Frag<Cfg<NT, CS>::KS> &a, const uint16_t *Pth, const uint16_t *Ptl,
                                      const Geo &g, const Own<NT, CS> &o, f32x4 (&acc)[Own<NT, CS>::NIT])
{
    const int pt = g.npc + kBf2Pad, ks = g.npc / 32;
    // column tiles in pairs: two independent accumulator chains per k-step
#pragma unroll
    for (int v = 0; v < Own<NT, CS>::NIT; v += 2) {
        if (o.v0 + v >= o.nti) break;
        const bool two = v + 1 < Own<NT, CS>::NIT;
        const int e0 = o.col(v) * pt + 8 * o.lq, e1 = e0 + 16 * pt;
#pragma unroll
        for (int s = 0; s < Cfg<NT, CS>::KS; ++s) {
            if (s >= ks) break;
            const bf16x8 b0h = ld8(Pth + e0 + 32 * s), b0l = ld8(Ptl + e0 + 32 * s);
            if (two) {
                const bf16x8 b1h = ld8(Pth + e1 + 32 * s), b1l = ld8(Ptl + e1 + 32 * s);
                acc[v] = mma_bf(a.h[s], b0h, acc[v]);
                acc[v + two] = mma_bf(a.h[s], b1h, acc[v + two]);
                acc[v] = mma_bf(a.h[s], b0l, acc[v]);
                acc[v + two] = mma_bf(a.h[s], b1l, acc[v + two]);
                acc[v] = mma_bf(a.l[s], b0h, acc[v]);
                acc[v + two] = mma_bf(a.l[s], b1h, acc[v + two]);
            } else {
                acc[v] = mma_bf(a.h[s], b0h, acc[v]);
                acc[v] = mma_bf(a.h[s], b0l, acc[v]);
                acc[v] = mma_bf(a.l[s], b0h, acc[v]);
            }
        }
    }
}

// The along-i matrix of a contraction, B(k, i) = M[i][k] with M row-major:
// held fragments of the wave's column tiles, or the matrix itself.
template <int NT, int CS> struct MatI {
    const uint16_t *h, *l;
    Frag<Cfg<NT, CS>::HOLD ? Cfg<NT, CS>::KS : 1> f[Cfg<NT, CS>::HOLD ? Own<NT, CS>::NIT : 1];
    __device__ __forceinline__ MatI(const uint16_t *Mh, const uint16_t *Ml) : h(Mh), l(Ml) {}
    __device__ __forceinline__ void load(const Geo &g, const Own<NT, CS> &o)
    {
        if constexpr (Cfg<NT, CS>::HOLD) {
#pragma unroll
            for (int v = 0; v < Own<NT, CS>::NIT; ++v)
                f[v].load(glb(h), glb(l), g.npi, o.v0 + v < o.nti ? o.v0 + v : 0, o.l16, o.lq, g.npi / 32);
        }
    }
};

// acc(c, i) += sum_k P[c][k] M[k][i]: A = the wave's rows of the c-major plane
template <int NT, int CS>
__device__ __forceinline__ void mul_i(const uint16_t *Pch, const uint16_t *Pcl, const MatI<NT, CS> &m,
                                      const Geo &g, const Own<NT, CS> &o, f32x4 (&acc)[Own<NT, CS>::NIT])
{
    constexpr int KS = Cfg<NT, CS>::KS;
    const int ks = g.npi / 32;
    Frag<KS> a;
    a.load(Pch, Pcl, g.npi + kBf2Pad, o.tc, o.l16, o.lq, ks);
#pragma unroll
    for (int v = 0; v < Own<NT, CS>::NIT; ++v) {
        if (o.v0 + v >= o.nti) break;
        if constexpr (Cfg<NT, CS>::HOLD) {
            mm(a, m.f[v], ks, acc[v]);
        } else {
            Frag<KS> b;
            b.load(glb(m.h), glb(m.l), g.npi, o.v0 + v, o.l16, o.lq, ks);
            mm(a, b, ks, acc[v]);
        }
    }
}

template <int N> __device__ __forceinline__ void zero(f32x4 (&acc)[N])
{
#pragma unroll
    for (int v = 0; v < N; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
}

template <typename D> __device__ __forceinline__ D of_f32(float v) { return (D)v; }
template <> __device__ __forceinline__ uint16_t of_f32<uint16_t>(float v) { return bf16_rne(v); }

// Stores the owned tiles to FP64, FP32 or BF16 (uint16_t bit patterns, rounded
// to nearest even) storage.
template <typename D, int NT, int CS>
__device__ __forceinline__ void own_store(D *dst, const Geo &g, const Own<NT, CS> &o,
                                          const f32x4 (&acc)[Own<NT, CS>::NIT])
{
    const gptr<D> d = glb(dst) + g.base;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = o.row(r);
        const unsigned oc = (unsigned)c * (unsigned)g.cs;
#pragma unroll
        for (int v = 0; v < Own<NT, CS>::NIT; ++v)
            if (c < g.nc && o.col(v) < g.ni)
                *reinterpret_cast<gptr<D>>(reinterpret_cast<gptr<char>>(d) +
                                           (oc + (unsigned)o.col(v)) * (unsigned)sizeof(D)) = of_f32<D>(acc[v][r]);
    }
}

// ------------------------------------------------------------------ H*X, split-BF16 form
// Pass A (plane (i,j) at k): Y = V o X + Ty X along c = j; the accumulators
// start from V o X.  Pass B (plane (i,k) at j): Y += Tz X along c = k + X Tx
// along i.  LDS: the i-major plane (pass A), plus the c-major plane (pass B).
// Plane p of job J; returns at once where p is past the job's planes.
template <int PASS, int NT, int CS>
__device__ __forceinline__ void hx_bf2_plane(const HxJob &J, int p, unsigned char *smem)
{
    constexpr int NIT = Own<NT, CS>::NIT;
    const AxisMats &Mi = J.ax[0];
    const AxisMats &Mc = J.ax[PASS == 0 ? 1 : 2];
    Geo g;
    if (!geo_of(PASS, J.nx, J.ny, J.nz, J.nvec, J.ld, Mi.np, Mc.np, p, g)) return;
    const Own<NT, CS> o(g);
    const int pt = g.npc + kBf2Pad, pc = g.npi + kBf2Pad;
    uint16_t *Pth = reinterpret_cast<uint16_t *>(smem);
    uint16_t *Ptl = Pth + g.npi * pt;
    uint16_t *Pch = Ptl + g.npi * pt;
    uint16_t *Pcl = Pch + g.npc * pc;
    float *Y = static_cast<float *>(J.Y);
    const float *W = PASS == 0 ? static_cast<const float *>(J.V) : Y;  // V (pass A) or Y (pass B)
    float xb[NIT][4], wb[NIT][4];
    Frag<Cfg<NT, CS>::KS> a;
    MatI<NT, CS> ti(Mi.th, Mi.tl);  // B(k, i) = Tx[k][i] = Tx[i][k] (symmetric)
    own_load<float, NT, CS>(static_cast<const float *>(J.X), g.base, g, o, xb);
    if (o.active) {
        a.load(glb(Mc.th), glb(Mc.tl), g.npc, o.tc, o.l16, o.lq, g.npc / 32);
        if (PASS == 1) ti.load(g, o);
        own_load<float, NT, CS>(W, PASS == 0 ? g.vbase : g.base, g, o, wb);
    }
    own_put<NT, CS>(xb, g, o, Pth, Ptl, PASS == 1 ? Pch : nullptr, Pcl);
    __syncthreads();
    if (!o.active) return;
    f32x4 acc[NIT];
#pragma unroll
    for (int v = 0; v < NIT; ++v)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[v][r] = PASS == 0 ? wb[v][r] * xb[v][r] : 0.f;
    mul_c<NT, CS>(a, Pth, Ptl, g, o, acc);
    if (PASS == 1) {
        mul_i<NT, CS>(Pch, Pcl, ti, g, o, acc);
#pragma unroll
        for (int v = 0; v < NIT; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[v][r] = wb[v][r] + acc[v][r];
    }
    own_store<float, NT, CS>(Y, g, o, acc);
}

template <int PASS, int NT, int CS>
__global__ void __launch_bounds__((Cfg<NT, CS>::THREADS), (CS == 1 ? 4 : 1)) hx_bf2_kernel(const HxJob *__restrict__ jobs)
{
    extern __shared__ __align__(16) unsigned char smem[];
    hx_bf2_plane<PASS, NT, CS>(jobs[plane_y(PASS == 1)], plane_x(PASS == 1), smem);
}

template <int PASS, int NT, int CS>
__global__ void __launch_bounds__((Cfg<NT, CS>::THREADS), (CS == 1 ? 4 : 1)) hx_bf2_one_kernel(HxJob J)
{
    extern __shared__ __align__(16) unsigned char smem[];
    hx_bf2_plane<PASS, NT, CS>(J, plane_x(PASS == 1), smem);
}

// ------------------------------------------------------------------ H*X, split-BF16, one launch
// Both passes in one launch, ordered per XCD so that pass B of a vector reads
// the X and Y that pass A left in that XCD's L2 instead of HBM.  The vectors
// are split into eight contiguous runs of about equal work, one per XCD; the
// workgroups of an XCD (read from the hardware's XCC_ID) take tickets from
// that XCD's counter in order, `batch` consecutive tickets per counter
// increment (one atomic per ticket serialised the 64 workgroups of an XCD on
// the counter's cache line: ~0.5 us per draw), each batch worked through in
// order, and the ticket sequence of run s0, s1, ... is
//   A(s0) | A(s1) B(s0) | A(s2) B(s1) | ... | B(s_last)
// (A(s): the n_z (i,j) planes of pass A of vector s; B(s): its n_y (i,k)
// planes).  A workgroup that draws a plane of B(s) waits until every plane
// of A(s) is stored: each A plane, once its stores have completed (all
// memory counters drained), adds 1 to the vector's completion count, and the
// wait polls that count in the XCD's L2.  Every plane a ticket waits on has a
// smaller ticket: either earlier in the waiting workgroup's own batch (done
// already) or drawn earlier by a running workgroup, which works through its
// batch in order and can itself wait only on smaller tickets; the smallest
// unfinished ticket waits on nothing, so the wait always ends.  It is bounded
// all the same (a spin limit; a workgroup past it counts the event in
// hx_spin_timeouts and goes on).
// X is not written by the launch and Y of a vector only by its own A and B
// planes, so no stale copy of either can sit in a CU's L1: the L1 is written
// through and holds only lines that the CU read after their last writer
// finished.
// Plan layout (ints): [0, 8) ticket counters, [8, 16) tickets per XCD,
// [16, 25) first segment of each XCD, [25] number of vectors, then the
// vectors' completion counts, then the segments (kSegInts ints each:
// job, vector, pass, first ticket, planes, vector slot).  The counters arrive
// zeroed with the plan.
constexpr int kSegInts = 6;
constexpr int kXcds = 8;
__device__ unsigned int hx_spin_timeouts;

// The ticket and completion counters of an XCD are touched only by that XCD's
// workgroups, and read-modify-writes are performed in the L2 (the vector L1
// performs no atomics), which every CU of the XCD shares.  A count is read by
// a compare-and-swap that never matches (an atomic performed in the L2), not
// by a load: a workgroup-scope load may be served by the L1, and an atomic add
// of 0 is compiled as such a load.
__device__ __forceinline__ int xcd_add(int *p, int v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int xcd_read(int *p)
{
    int seen = -1;  // counts are never negative: the swap never happens
    __hip_atomic_compare_exchange_strong(p, &seen, -1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
    return seen;
}

template <int NT>
__global__ void __launch_bounds__((Cfg<NT, 2>::THREADS)) hx_bf2_fused_kernel(const HxJob *__restrict__ jobs,
                                                           int *__restrict__ plan, int batch)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_task[4];  // job, vector, pass, plane; -1 job: no tickets left
    const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & (kXcds - 1);
    const int nvecs = plan[25];
    int *done = plan + 26;
    const int *segs = plan + 26 + nvecs;
    const int seg_end = plan[16 + xcc + 1];
    int cursor = plan[16 + xcc];
    int bt = 0, be = 0;  // thread 0: the next ticket of the workgroup's batch, its end
    for (;;) {
        if (threadIdx.x == 0) {
            if (bt >= be) {
                bt = xcd_add(plan + xcc, batch);
                be = bt + batch;
            }
            const int t = bt++;
            int job = -1;
            if (t < plan[8 + xcc]) {
                while (cursor < seg_end && t >= segs[kSegInts * cursor + 3] + segs[kSegInts * cursor + 4])
                    ++cursor;
                const int *sg = segs + kSegInts * cursor;
                job = sg[0];
                s_task[1] = sg[1];
                s_task[2] = sg[2];
                s_task[3] = t - sg[3];
                if (sg[2] == 1) {
                    // pass B: every (i,j) plane of this vector's pass A must be stored
                    const int need = jobs[sg[0]].nz;
                    unsigned spins = 0;
                    while (xcd_read(done + sg[5]) < need) {
                        __builtin_amdgcn_s_sleep(2);
                        if (++spins > (1u << 24)) {
                            atomicAdd(&hx_spin_timeouts, 1u);
                            break;
                        }
                    }
                }
            }
            s_task[0] = job;
        }
        __syncthreads();
        const int job = s_task[0];
        if (job < 0) break;
        const HxJob &J = jobs[job];
        const int pass = s_task[2];
        // plane index within the job: vector-major, as the two-launch kernels count
        if (pass == 0) hx_bf2_plane<0, NT, 2>(J, s_task[1] * J.nz + s_task[3], smem);
        else hx_bf2_plane<1, NT, 2>(J, s_task[1] * J.ny + s_task[3], smem);
        if (pass == 0) {
            // this plane's Y stores have reached the L2 before it is counted
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (threadIdx.x == 0) {
                const int *sg = segs + kSegInts * cursor;
                xcd_add(done + sg[5], 1);
            }
        }
        __syncthreads();  // s_task and the LDS planes are reused by the next ticket
    }
}

// ------------------------------------------------------------------ preconditioner, split-BF16
// Three passes, one plane per workgroup as H*X:
//   0, plane (i,j) at k: r -> c-major plane; X Qx along i -> i-major plane;
//      Qy^T (.) along c -> work
//   1, plane (i,k) at j: work -> i-major plane A; Qz^T (.) along c, scaled by
//      scale / (lam_x[i] + lam_y[j] - shift + lam_z[c]) (formed in FP32: the
//      scaled values are FP32 and go on as split BF16) -> i-major plane B;
//      Qz (.) along c -> work
//   2, plane (i,j) at k: work -> i-major plane; Qy (.) along c -> c-major
//      plane; (.) Qx^T along i -> t
// Plane p, or with MULTI the planes p, p + pstride, ... of one pass of task t:
// the matrix fragments are then fetched once for several planes and the next
// plane is requested before the current one is contracted.
template <int PASS, int NT, int CS, bool MULTI>
__device__ __forceinline__ void fdm_bf2_plane(const FdmTask &t, int p, int pstride, unsigned char *smem)
{
    constexpr int NIT = Own<NT, CS>::NIT, KS = Cfg<NT, CS>::KS;
    const AxisMats &Mx = t.ax[0], &My = t.ax[1], &Mz = t.ax[2];
    const AxisMats &Mc = PASS == 1 ? Mz : My;
    Geo g;
    if (!geo_of(PASS == 1 ? 1 : 0, Mx.n, My.n, Mz.n, 1, 0, Mx.np, Mc.np, p, g)) return;
    const Own<NT, CS> o(g);
    const int pt = g.npc + kBf2Pad, pc = g.npi + kBf2Pad, ksc = g.npc / 32;
    uint16_t *Pth = reinterpret_cast<uint16_t *>(smem);
    uint16_t *Ptl = Pth + g.npi * pt;
    uint16_t *P2h = Ptl + g.npi * pt;  // c-major plane (passes 0, 2) or i-major plane B (pass 1)
    uint16_t *P2l = P2h + (PASS == 1 ? g.npi * pt : g.npc * pc);
    float xb[NIT][4], lx[NIT], lz[4];
    Frag<KS> a, b;
    // B form of Qx (pass 0) and of Qx^T (pass 2)
    MatI<NT, CS> mi(PASS == 0 ? Mx.qth : Mx.qh, PASS == 0 ? Mx.qtl : Mx.ql);
    // pass 0 reads r (FP64 or FP32); passes 1 and 2 the BF16 intermediate
    auto load = [&](const Geo &gg) {
        if constexpr (PASS != 0) own_load<uint16_t, NT, CS>(static_cast<const uint16_t *>(t.work), gg.base, gg, o, xb);
        else if (t.src32) own_load<float, NT, CS>(static_cast<const float *>(t.src), gg.base, gg, o, xb);
        else own_load<double, NT, CS>(static_cast<const double *>(t.src), gg.base, gg, o, xb);
    };
    load(g);
    if (o.active) {
        // along c: Qy^T (pass 0), Qz^T then Qz (pass 1), Qy (pass 2)
        a.load(glb(PASS == 2 ? My.qh : Mc.qth), glb(PASS == 2 ? My.ql : Mc.qtl), g.npc, o.tc, o.l16, o.lq, ksc);
        if (PASS == 1) {
            if (NT < 8) b.load(glb(Mz.qh), glb(Mz.ql), g.npc, o.tc, o.l16, o.lq, ksc);
#pragma unroll
            for (int v = 0; v < NIT; ++v) lx[v] = (float)at<double>(glb(Mx.lam), o.col(v) < g.ni ? o.col(v) : 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) lz[r] = (float)at<double>(glb(Mz.lam), o.row(r) < g.nc ? o.row(r) : 0);
        } else {
            mi.load(g, o);
        }
    }
    const float scale = (float)t.scale, floor = (float)t.floor;
    for (;;) {
        const double ly = PASS == 1 ? glb(My.lam)[g.pl] : 0.0;
        own_put<NT, CS>(xb, g, o, PASS == 0 ? nullptr : Pth, Ptl, PASS == 0 ? P2h : nullptr, P2l);
        __syncthreads();
        Geo gn;
        const bool more = MULTI && geo_of(PASS == 1 ? 1 : 0, Mx.n, My.n, Mz.n, 1, 0, Mx.np, Mc.np, p + pstride, gn);
        if (more) load(gn);
        f32x4 acc[NIT];
        zero(acc);
        if (o.active) {
            if (PASS == 0) mul_i<NT, CS>(P2h, P2l, mi, g, o, acc);  // X Qx
            else mul_c<NT, CS>(a, Pth, Ptl, g, o, acc);             // Qz^T X, Qy X
            // both matrices at once exceed the registers of 16 waves
            if (PASS == 1 && NT == 8) b.load(glb(Mz.qh), glb(Mz.ql), g.npc, o.tc, o.l16, o.lq, ksc);
        }
        const float fly = (float)(ly - t.shift);
        float y[NIT][4];
#pragma unroll
        for (int v = 0; v < NIT; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (PASS == 1) {
                    // outside the plane the accumulators are 0
                    float den = o.active && o.col(v) < g.ni && o.row(r) < g.nc ? lx[v] + fly + lz[r] : 1.f;
                    if (t.absden) den = fabsf(den);
                    if (fabsf(den) < floor) den = den < 0.f ? -floor : floor;
                    y[v][r] = acc[v][r] * (scale / den);
                } else {
                    y[v][r] = acc[v][r];
                }
            }
        // the other plane's LDS: its last readers are past the barrier above
        if (PASS == 0) own_put<NT, CS>(y, g, o, Pth, Ptl, nullptr, nullptr);
        else if (PASS == 1) own_put<NT, CS>(y, g, o, P2h, P2l, nullptr, nullptr);
        else own_put<NT, CS>(y, g, o, nullptr, nullptr, P2h, P2l);
        __syncthreads();
        if (o.active) {
            zero(acc);
            if (PASS == 0) mul_c<NT, CS>(a, Pth, Ptl, g, o, acc);        // Qy^T (.)
            else if (PASS == 1) mul_c<NT, CS>(b, P2h, P2l, g, o, acc);   // Qz (.)
            else mul_i<NT, CS>(P2h, P2l, mi, g, o, acc);                 // (.) Qx^T
            if (PASS != 2) own_store<uint16_t, NT, CS>(t.work, g, o, acc);
            else if (t.dst32) own_store<float, NT, CS>(static_cast<float *>(t.dst), g, o, acc);
            else own_store<double, NT, CS>(static_cast<double *>(t.dst), g, o, acc);
        }
        if (!more) break;
        g = gn;
        p += pstride;
    }
}

template <int PASS, int NT, int CS, bool MULTI>
__global__ void __launch_bounds__((Cfg<NT, CS>::THREADS)) fdm_bf2_kernel(const FdmTask *__restrict__ tasks)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fdm_bf2_plane<PASS, NT, CS, MULTI>(tasks[plane_y(PASS == 1)], plane_x(PASS == 1), gridDim.x, smem);
}

template <int PASS, int NT, int CS, bool MULTI>
__global__ void __launch_bounds__((Cfg<NT, CS>::THREADS)) fdm_bf2_one_kernel(FdmOne one)
{
    extern __shared__ __align__(16) unsigned char smem[];
    fdm_bf2_plane<PASS, NT, CS, MULTI>(task_of(one, plane_y(PASS == 1), one.t.src32 ? 4 : 8, one.t.dst32 ? 4 : 8),
                                       plane_x(PASS == 1), gridDim.x, smem);
}

// ------------------------------------------------------------------ preconditioner, one launch
// The three passes of the split-BF16 preconditioner in one launch, ordered per
// XCD as the one-launch H*X is: the vectors split into eight contiguous runs,
// one per XCD, whose ticket sequence is
//   P0(s0) | P0(s1) P1(s0) | P0(s2) P1(s1) P2(s0) | ... | P2(s_last)
// so that pass 1 reads the intermediate pass 0 left in the XCD's L2 and pass 2
// the one pass 1 left there.  A plane of P1(s) waits until every plane of
// P0(s) is stored, a plane of P2(s) until every plane of P1(s) is; the counts
// are kept per vector as for H*X, and every awaited plane was drawn earlier by
// a resident workgroup that is not waiting on a later one.
// Plan layout (ints): [0, 8) ticket counters, [8, 16) tickets per XCD,
// [16, 25) first segment of each XCD, [25] vectors, then per vector the
// completion counts of pass 0 and of pass 1, then the segments (task, 0,
// pass, first ticket, planes, vector slot).
template <int NT>
__global__ void __launch_bounds__((Cfg<NT, 2>::THREADS)) fdm_bf2_fused_kernel(const FdmTask *__restrict__ tasks,
                                                            int *__restrict__ plan, int batch)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_task[3];  // task, pass, plane; -1 task: no tickets left
    const unsigned xcc = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & (kXcds - 1);
    const int nvecs = plan[25];
    int *done = plan + 26;  // done[2 v + pass]
    const int *segs = plan + 26 + 2 * nvecs;
    const int seg_end = plan[16 + xcc + 1];
    int cursor = plan[16 + xcc];
    int bt = 0, be = 0;  // thread 0: the next ticket of the workgroup's batch, its end
    for (;;) {
        if (threadIdx.x == 0) {
            if (bt >= be) {
                bt = xcd_add(plan + xcc, batch);
                be = bt + batch;
            }
            const int t = bt++;
            int task = -1;
            if (t < plan[8 + xcc]) {
                while (cursor < seg_end && t >= segs[kSegInts * cursor + 3] + segs[kSegInts * cursor + 4])
                    ++cursor;
                const int *sg = segs + kSegInts * cursor;
                task = sg[0];
                s_task[1] = sg[2];
                s_task[2] = t - sg[3];
                if (sg[2] > 0) {
                    // every plane of the previous pass of this vector must be stored
                    const FdmTask &T = tasks[sg[0]];
                    const int need = sg[2] == 1 ? T.ax[2].n : T.ax[1].n;
                    unsigned spins = 0;
                    while (xcd_read(done + 2 * sg[5] + sg[2] - 1) < need) {
                        __builtin_amdgcn_s_sleep(2);
                        if (++spins > (1u << 24)) {
                            atomicAdd(&hx_spin_timeouts, 1u);
                            break;
                        }
                    }
                }
            }
            s_task[0] = task;
        }
        __syncthreads();
        const int task = s_task[0];
        if (task < 0) break;
        const FdmTask &T = tasks[task];
        const int pass = s_task[1];
        if (pass == 0) fdm_bf2_plane<0, NT, 2, false>(T, s_task[2], 1, smem);
        else if (pass == 1) fdm_bf2_plane<1, NT, 2, false>(T, s_task[2], 1, smem);
        else fdm_bf2_plane<2, NT, 2, false>(T, s_task[2], 1, smem);
        if (pass < 2) {
            // this plane's stores have reached the L2 before it is counted
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (threadIdx.x == 0) {
                const int *sg = segs + kSegInts * cursor;
                xcd_add(done + 2 * sg[5] + pass, 1);
            }
        }
        __syncthreads();  // s_task and the LDS planes are reused by the next ticket
    }
}

// ------------------------------------------------------------------ launch helpers
size_t bf2_lds(int np) { return (size_t)2 * 2 * np * (np + kBf2Pad) * sizeof(uint16_t); }

// a positive integer from the environment, else def
int env_or(const char *env, int def)
{
    const char *e = std::getenv(env);
    const int v = e ? std::atoi(e) : 0;
    return v > 0 ? v : def;
}

template <int NT, int CS>
void hx_bf2_launch(const HxJob *d, const HxJob *one, int n, int pa, int pb, hipStream_t s)
{
    static std::once_flag once;
    std::call_once(once, [] {
        allow_lds(hx_bf2_kernel<0, NT, CS>);
        allow_lds(hx_bf2_kernel<1, NT, CS>);
        allow_lds(hx_bf2_one_kernel<0, NT, CS>);
        allow_lds(hx_bf2_one_kernel<1, NT, CS>);
    });
    const size_t lds = bf2_lds(16 * NT);
    const dim3 blk(Cfg<NT, CS>::THREADS);
    // pass A uses only the i-major plane (first half of the layout)
    if (one) {
        hipLaunchKernelGGL((hx_bf2_one_kernel<0, NT, CS>), dim3(pa), blk, lds / 2, s, *one);
        hipLaunchKernelGGL((hx_bf2_one_kernel<1, NT, CS>), dim3(pb), blk, lds, s, *one);
        return;
    }
    hipLaunchKernelGGL((hx_bf2_kernel<0, NT, CS>), dim3(pa, n), blk, lds / 2, s, d);
    hipLaunchKernelGGL((hx_bf2_kernel<1, NT, CS>), dim3(pb, n), blk, lds, s, d);
}

template <int NT, int CS, bool MULTI>
void fdm_bf2_launch(const FdmTask *d, const FdmOne *one, int n, int nplanes, hipStream_t s, int ppw = 1)
{
    static std::once_flag once;
    std::call_once(once, [] {
        allow_lds(fdm_bf2_kernel<0, NT, CS, MULTI>);
        allow_lds(fdm_bf2_kernel<1, NT, CS, MULTI>);
        allow_lds(fdm_bf2_kernel<2, NT, CS, MULTI>);
        allow_lds(fdm_bf2_one_kernel<0, NT, CS, MULTI>);
        allow_lds(fdm_bf2_one_kernel<1, NT, CS, MULTI>);
        allow_lds(fdm_bf2_one_kernel<2, NT, CS, MULTI>);
    });
    const size_t lds = bf2_lds(16 * NT);
    const dim3 grid((nplanes + ppw - 1) / ppw, n), blk(Cfg<NT, CS>::THREADS);
    if (one) {
        hipLaunchKernelGGL((fdm_bf2_one_kernel<0, NT, CS, MULTI>), grid, blk, lds, s, *one);
        hipLaunchKernelGGL((fdm_bf2_one_kernel<1, NT, CS, MULTI>), grid, blk, lds, s, *one);
        hipLaunchKernelGGL((fdm_bf2_one_kernel<2, NT, CS, MULTI>), grid, blk, lds, s, *one);
        return;
    }
    hipLaunchKernelGGL((fdm_bf2_kernel<0, NT, CS, MULTI>), grid, blk, lds, s, d);
    hipLaunchKernelGGL((fdm_bf2_kernel<1, NT, CS, MULTI>), grid, blk, lds, s, d);
    hipLaunchKernelGGL((fdm_bf2_kernel<2, NT, CS, MULTI>), grid, blk, lds, s, d);
}

}  // namespace

namespace {
void hx_dispatch(const HxJob *d_jobs, const HxJob *one, int njobs, int max_planes_a, int max_planes_b,
                 int max_n, int precision, hipStream_t s)
{
    if (njobs <= 0) return;
    PC_REQUIRE(max_n > 0 && max_n <= 128, PISCES_ERR_UNSUPPORTED, "grid dimension above 128");
    if (precision != PISCES_BF16X2) {
        hx_f_launch(d_jobs, one, njobs, max_planes_a, max_planes_b, max_n, precision, s);
        return;
    }
    const int np = axis_pad(max_n);
    if (np <= 32) hx_bf2_launch<2, 2>(d_jobs, one, njobs, max_planes_a, max_planes_b, s);
    else if (np <= 64) {
        // Few planes: eight waves each, for the latency of a plane; more than
        // about 1.5 a CU: four waves and fewer registers, so that four planes
        // are in flight on a CU instead of two.  us at 64^3, eight / four waves:
        // 4 vectors 14.4 / 15.2, 8 20.8 / 20.1, 32 49.9 / 47.8, 128 161 / 147;
        // at 48^3 128 vectors 102 / 75.
        if ((long long)njobs * max_planes_a < 384)
            hx_bf2_launch<4, 2>(d_jobs, one, njobs, max_planes_a, max_planes_b, s);
        else
            hx_bf2_launch<4, 1>(d_jobs, one, njobs, max_planes_a, max_planes_b, s);
    }
    else if (np <= 96) hx_bf2_launch<6, 2>(d_jobs, one, njobs, max_planes_a, max_planes_b, s);
    else hx_bf2_launch<8, 2>(d_jobs, one, njobs, max_planes_a, max_planes_b, s);
    PC_HIP(hipGetLastError());
}
}  // namespace

void hx_mfma_launch(const HxJob *d_jobs, int njobs, int max_planes_a, int max_planes_b, int max_n,
                    int precision, hipStream_t s)
{
    hx_dispatch(d_jobs, nullptr, njobs, max_planes_a, max_planes_b, max_n, precision, s);
}

void hx_launch_one(const HxJob &J, int precision, hipStream_t s)
{
    hx_dispatch(nullptr, &J, 1, J.nz * J.nvec, J.ny * J.nvec, std::max(J.nx, std::max(J.ny, J.nz)), precision, s);
}

int hx_fused_plan_ints(const HxJob *h_jobs, int njobs)
{
    int nv = 0;
    for (int j = 0; j < njobs; ++j) nv += h_jobs[j].nvec;
    return 26 + nv + kSegInts * 2 * nv;
}

void hx_fused_plan(const HxJob *h_jobs, int njobs, int *plan)
{
    // every vector (job-major) with its plane work; eight contiguous runs of
    // about equal work, one per XCD, so the vectors of a job mostly share an
    // XCD and its L2 copy of the job's potential
    struct Vec { int job, vec; double w; };
    std::vector<Vec> vs;
    double total = 0;
    for (int j = 0; j < njobs; ++j) {
        const HxJob &J = h_jobs[j];
        const double w = (double)(J.nz + J.ny) * axis_pad(J.nx) * axis_pad(std::max(J.ny, J.nz));
        for (int v = 0; v < J.nvec; ++v) {
            vs.push_back({j, v, w});
            total += w;
        }
    }
    const int nv = (int)vs.size();
    std::fill(plan, plan + 26 + nv, 0);
    plan[25] = nv;
    int *segs = plan + 26 + nv;
    int nseg = 0, k = 0;
    double acc = 0;
    for (int x = 0; x < kXcds; ++x) {
        plan[16 + x] = nseg;
        std::vector<int> run;  // vector indices of this XCD, in order
        const double upto = total * (x + 1) / kXcds;
        while (k < nv && (x == kXcds - 1 || acc + 0.5 * vs[k].w <= upto)) {
            acc += vs[k].w;
            run.push_back(k++);
        }
        int t = 0;
        auto add = [&](int vi, int pass) {
            const HxJob &J = h_jobs[vs[vi].job];
            int *sg = segs + kSegInts * nseg++;
            sg[0] = vs[vi].job;
            sg[1] = vs[vi].vec;
            sg[2] = pass;
            sg[3] = t;
            sg[4] = pass == 0 ? J.nz : J.ny;
            sg[5] = vi;
            t += sg[4];
        };
        // A(s0) | A(s1) B(s0) | ... | B(s_last)
        for (size_t r = 0; r < run.size(); ++r) {
            add(run[r], 0);
            if (r > 0) add(run[r - 1], 1);
        }
        if (!run.empty()) add(run.back(), 1);
        plan[8 + x] = t;
    }
    plan[16 + kXcds] = nseg;
}

namespace {
template <int NT>
void hx_fused_nt_launch(const HxJob *d_jobs, int *d_plan, int max_tickets, hipStream_t s)
{
    static std::once_flag once;
    std::call_once(once, [] { allow_lds(hx_bf2_fused_kernel<NT>, bf2_lds(16 * NT)); });
    // workgroups per XCD: two per CU (32 CUs) unless an XCD has fewer planes
    static const int wpx = env_or("PISCES_HXF_WG", 64);
    static const int batch = env_or("PISCES_HXF_BATCH", 4);
    const int w = std::max(1, std::min(wpx, max_tickets));
    hipLaunchKernelGGL((hx_bf2_fused_kernel<NT>), dim3(kXcds * w), dim3(Cfg<NT, 2>::THREADS), bf2_lds(16 * NT), s,
                       d_jobs, d_plan, batch);
}
}  // namespace

void hx_fused_launch(const HxJob *h_jobs, const HxJob *d_jobs, int njobs, const int *h_plan,
                     int *d_plan, int max_n, hipStream_t s)
{
    if (njobs <= 0) return;
    PC_REQUIRE(max_n > 0 && max_n <= 128, PISCES_ERR_UNSUPPORTED, "grid dimension above 128");
    int mt = 0;
    for (int x = 0; x < kXcds; ++x) mt = std::max(mt, h_plan[8 + x]);
    const int np = axis_pad(max_n);
    if (np <= 32) hx_fused_nt_launch<2>(d_jobs, d_plan, mt, s);
    else if (np <= 64) hx_fused_nt_launch<4>(d_jobs, d_plan, mt, s);
    else hx_fused_nt_launch<8>(d_jobs, d_plan, mt, s);
    PC_HIP(hipGetLastError());
}

bool one_launch_available()
{
    // the ordering needs the eight XCDs of one device (SPX partitioning):
    // with fewer compute units the device is a partition of one XCD
    static const bool on = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return false;
        return cus >= 8 * 16;
    }();
    return on;
}

// The one-launch forms are opt-in (PISCES_HX_FUSED=1, PISCES_FDM_FUSED=1): at
// 64^3 x 64 vectors they take 0.296 ms (H*X) and 0.442 ms (preconditioner)
// against 0.081 and 0.121 ms for the multi-launch forms.  An XCD keeps 64 tickets
// (workgroups) in flight, so a ticket of its 1024 (1536) takes about 18 us from
// draw to counted store, where the multi-launch grids keep thousands of planes
// going; these kernels are bound by that latency, not by the HBM traffic the L2
// reuse saves.
bool hx_fused_enabled()
{
    static const bool on = [] {
        const char *e = std::getenv("PISCES_HX_FUSED");
        return e && e[0] == '1' && one_launch_available();
    }();
    return on;
}

unsigned hx_fused_spin_timeouts()
{
    // a stream of its own (released again), not the null stream
    unsigned v = 0;
    hipStream_t s;
    PC_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    const hipError_t e = hipMemcpyFromSymbolAsync(&v, HIP_SYMBOL(hx_spin_timeouts), sizeof(v), 0,
                                                  hipMemcpyDeviceToHost, s);
    const hipError_t w = hipStreamSynchronize(s);
    static_cast<void>(hipStreamDestroy(s));
    PC_HIP(e);
    PC_HIP(w);
    return v;
}

int fdm_fused_plan_ints(int ntasks) { return 26 + 2 * ntasks + kSegInts * 3 * ntasks; }

void fdm_fused_plan(const FdmTask *h_tasks, int ntasks, int *plan)
{
    // runs of about equal work per XCD (plane work ~ planes x plane size)
    std::vector<double> w(ntasks);
    double total = 0;
    for (int i = 0; i < ntasks; ++i) {
        const FdmTask &T = h_tasks[i];
        w[i] = (double)(2 * T.ax[2].n + T.ax[1].n) * axis_pad(T.ax[0].n) *
               axis_pad(std::max(T.ax[1].n, T.ax[2].n));
        total += w[i];
    }
    std::fill(plan, plan + 26 + 2 * ntasks, 0);
    plan[25] = ntasks;
    int *segs = plan + 26 + 2 * ntasks;
    int nseg = 0, k = 0;
    double acc = 0;
    for (int x = 0; x < kXcds; ++x) {
        plan[16 + x] = nseg;
        std::vector<int> run;
        const double upto = total * (x + 1) / kXcds;
        while (k < ntasks && (x == kXcds - 1 || acc + 0.5 * w[k] <= upto)) {
            acc += w[k];
            run.push_back(k++);
        }
        int t = 0;
        auto add = [&](int ti, int pass) {
            const FdmTask &T = h_tasks[ti];
            int *sg = segs + kSegInts * nseg++;
            sg[0] = ti;
            sg[1] = 0;
            sg[2] = pass;
            sg[3] = t;
            sg[4] = pass == 1 ? T.ax[1].n : T.ax[2].n;
            sg[5] = ti;
            t += sg[4];
        };
        // P0(s) | P0(s+1) P1(s) | P0(s+2) P1(s+1) P2(s) | ...
        const int S = (int)run.size();
        for (int st = 0; st < S + 2; ++st) {
            if (st < S) add(run[st], 0);
            if (st >= 1 && st - 1 < S) add(run[st - 1], 1);
            if (st >= 2 && st - 2 < S) add(run[st - 2], 2);
        }
        plan[8 + x] = t;
    }
    plan[16 + kXcds] = nseg;
}

namespace {
template <int NT>
void fdm_fused_nt_launch(const FdmTask *d_tasks, int *d_plan, int max_tickets, hipStream_t s)
{
    static std::once_flag once;
    std::call_once(once, [] { allow_lds(fdm_bf2_fused_kernel<NT>, bf2_lds(16 * NT)); });
    static const int wpx = env_or("PISCES_FDMF_WG", 64);
    static const int batch = env_or("PISCES_FDMF_BATCH", 4);
    const int w = std::max(1, std::min(wpx, max_tickets));
    hipLaunchKernelGGL((fdm_bf2_fused_kernel<NT>), dim3(kXcds * w), dim3(Cfg<NT, 2>::THREADS), bf2_lds(16 * NT), s,
                       d_tasks, d_plan, batch);
}
}  // namespace

void fdm_fused_launch(const FdmTask *d_tasks, int *d_plan, const int *h_plan, int max_n,
                      hipStream_t s)
{
    PC_REQUIRE(max_n > 0 && max_n <= 128, PISCES_ERR_UNSUPPORTED, "grid dimension above 128");
    int mt = 0;
    for (int x = 0; x < kXcds; ++x) mt = std::max(mt, h_plan[8 + x]);
    if (mt == 0) return;
    const int np = axis_pad(max_n);
    if (np <= 32) fdm_fused_nt_launch<2>(d_tasks, d_plan, mt, s);
    else if (np <= 64) fdm_fused_nt_launch<4>(d_tasks, d_plan, mt, s);
    else fdm_fused_nt_launch<8>(d_tasks, d_plan, mt, s);
    PC_HIP(hipGetLastError());
}

bool fdm_fused_enabled()
{
    static const bool on = [] {
        const char *e = std::getenv("PISCES_FDM_FUSED");
        return e && e[0] == '1' && one_launch_available();
    }();
    return on;
}

namespace {
void fdm_dispatch(const FdmTask *d_tasks, const FdmOne *one, int ntasks, int max_n, int precision,
                  hipStream_t s)
{
    if (ntasks <= 0) return;
    PC_REQUIRE(max_n > 0 && max_n <= 128, PISCES_ERR_UNSUPPORTED, "grid dimension above 128");
    if (precision == PISCES_FP64) {
        fdm_f64_launch(d_tasks, one, ntasks, max_n, s);
        return;
    }
    const int np = axis_pad(max_n);
    // planes per pass: the largest of ny (pass 1) and nz (passes 0, 2) <= max_n
    if (np <= 32) {
        fdm_bf2_launch<2, 2, false>(d_tasks, one, ntasks, max_n, s);
    } else if (np <= 64) {
        // Planes per workgroup by the number of planes: a plane's three matrix
        // fragments are as many bytes from the L2 as six planes, so workgroups
        // keep them for several planes as soon as that leaves every CU busy.  us
        // at 64^3 with 1 / 2 / 4 / 8 planes: 4 vectors 20 / 26 / 38 / 62, 16
        // 54 / 45 / 46 / 70, 32 91 / 71 / 62 / 70, 128 327 / 241 / 203 / 186.
        // (32-point planes: one is best or the same up to 128 vectors; 96 and
        // 128 points do not hold the along-i matrix.)  PISCES_PPW_FDM overrides.
        const long long planes = (long long)ntasks * max_n;
        static const int ppw_env = env_or("PISCES_PPW_FDM", 0);
        const int ppw = ppw_env ? ppw_env : planes < 600 ? 1 : planes < 1800 ? 2 : planes < 4096 ? 4 : 8;
        if (ppw == 1) fdm_bf2_launch<4, 2, false>(d_tasks, one, ntasks, max_n, s);
        else fdm_bf2_launch<4, 2, true>(d_tasks, one, ntasks, max_n, s, ppw);
    }
    else if (np <= 96) fdm_bf2_launch<6, 2, false>(d_tasks, one, ntasks, max_n, s);
    else fdm_bf2_launch<8, 2, false>(d_tasks, one, ntasks, max_n, s);
    PC_HIP(hipGetLastError());
}
}  // namespace

void fdm_launch(const FdmTask *d_tasks, int ntasks, int max_n, int precision, hipStream_t s)
{
    fdm_dispatch(d_tasks, nullptr, ntasks, max_n, precision, s);
}

void fdm_launch_one(const FdmOne &one, int nvec, int precision, hipStream_t s)
{
    const AxisMats *ax = one.t.ax;
    fdm_dispatch(nullptr, &one, nvec, std::max(ax[0].n, std::max(ax[1].n, ax[2].n)), precision, s);
}

}  // namespace pisces
