// Radix pass kernels for gfx950: the drop-in transforms and the CKKS forms.
//
// A transform of length L = 2^n is a sequence of radix-2 stages, each one
// pairing positions p and p ^ 2^b for one position bit b:
//   MODE_STD_FWD  Cooley-Tukey, bits n-1 .. 0, twiddle tab[base + (p >> (b+1))]
//                 (ForwardCore, reference src/lib/fft.cu:11-152; base = 2^(n-1-b)
//                 for X^N+1, 0 for X^N-1, fft.cu:67-74)
//   MODE_STD_INV  Gentleman-Sande, bits 0 .. n-1, same twiddle index
//                 (InverseCore, fft.cu:154-260)
//   MODE_SPE_FWD  Cooley-Tukey, bits 0 .. n-1, twiddle tab[2^b + (p & (2^b-1))]
//                 (Special_ForwardCore, fft.cu:856-926)
//   MODE_SPE_INV  Gentleman-Sande, bits n-1 .. 0, same twiddle index
//                 (Special_InverseCore, fft.cu:727-854)
//
// One launch ("pass") applies the stages of K consecutive bits [blo, blo+K) to
// tiles of 2^LT elements, one workgroup each, 16 elements per thread held in
// registers from the first load to the last store.  Two tile shapes:
//   row tiles (COL = 0)     blo = 0: 2^LT consecutive elements, i.e. whole
//                           transforms (K = n) or 2^(LT-K) blocks of 2^K;
//   column tiles (COL = 1)  2^K rows (the pass bits) by 2^(LT-K) consecutive
//                           positions below blo.
// The K bits are taken in ceil(K/4) radix steps of 4, 3 or 2 bits; between
// two steps the tile is re-dealt among the threads through LDS.  The step on
// the top bits reads and writes consecutive elements per lane, so it works on
// global memory directly; only the step on bits [0, 4) of a row tile needs one
// more exchange on its global side.
//
// What bounds it: HBM or the last-level cache for large batches, and the
// latency of load, exchanges and store for a few tiles.  Hence
//   * double exchanges move the real and then the imaginary parts, so a tile
//     of 2^12 elements takes 32 KiB of LDS and 4 workgroups share a CU (one
//     loads while another computes; the former 64 KiB tile allowed 2);
//   * a radix-16 group loads 8 twiddles, half of them ahead of the exchange in
//     front of it, and the other 7 are quarter turns (15 dependent loads before);
//   * geometry is compile-time, so addresses are one base per thread plus
//     constants (XOR constants in LDS).
// Measured against run-time geometry with every element through LDS first and
// a table load per twiddle, forward us per call on one buffer repeated, and on
// buffers cycled beyond the last-level cache:
//   FP64  2^13 x 1  14.4 -> 11.2          2^15 x 128  77 -> 41, 79 -> 56
//         2^23 x 1  198 -> 100, 214 -> 136
//   FP32  2^13 x 1  11.5 ->  7.7          2^16 x  64  60 -> 24, 65 -> 31
//         2^20 x 8  114 -> 43, 119 -> 55
//   special FP64  2^15 x 512  241 -> 135, 275 -> 166 (6.5 TB/s over its two passes)
// Radix steps of at most 3 bits (one more exchange at 8 and 12 bits) were 2-10%
// slower throughout.
#pragma once

#include <type_traits>

#include "cplx.hpp"
#include "engine.hpp"

namespace gfa {

template <typename T> struct RadixArgs {
    int n;      // log2 transform length
    int blo;    // lowest bit of the pass (column tiles)
    int batch;  // transforms in the launch
    int nega;   // X^N+1 twiddle base (standard modes only)
    int do_scale;
    cplx<T> scale;
    const cplx<T>* tab;  // root-of-unity table (reference layout)
    const void* src;
    const void* src2;      // second operand (LD_MUL, LD_RR_PACK)
    const cplx<T>* ltab;   // twist table (LD_FOLD), inverse root table (LD_RR_PACK)
    long long src_stride;  // elements between transforms
    void* dst;
    const cplx<T>* stab;  // untwist table (ST_UNFOLD); first summand (ST_SUM_F64)
    long long dst_stride;
    double delta;      // LD_CKKS / ST_CKKS scale
    double inv_delta;  // its inverse if it is a power of two, else 0 (LD_CKKS)
};

constexpr int PASS_E = 4;  // log2 of the elements per thread

// Radix steps of K bits, in ascending bit order, the wider ones first (the
// special modes' quarter turns want no step that starts at bit 1 or 2).
__host__ __device__ constexpr int pass_steps(int K) { return (K + 3) / 4; }
__host__ __device__ constexpr int pass_step_bits(int K, int s)
{
    return K / pass_steps(K) + (s < K % pass_steps(K) ? 1 : 0);
}
__host__ __device__ constexpr int pass_step_q(int K, int s)
{
    int q = 0;
    for (int i = 0; i < s; i++) q += pass_step_bits(K, i);
    return q;
}

// log2 of the tile: 2^12 elements (256 threads) where 16 columns of float or
// 8 of double (128-byte rows) fit beside the pass bits, else 2^13.
template <typename T> __host__ __device__ constexpr int pass_tile(int col, int K)
{
    return col ? (K <= (sizeof(T) == 8 ? 9 : 8) ? 12 : 13) : (K <= 12 ? 12 : 13);
}

// LDS slot of tile element i (8-byte slots).  Linear over XOR, so the slot of
// a thread's element is its base's slot XOR a constant; the three folds keep
// the lanes of (almost) every access of every step on distinct banks.
__host__ __device__ constexpr int slot_of(int i)
{
    return i ^ ((i >> 4) & 30) ^ ((i >> 7) & 31) ^ ((i >> 3) & 28);
}

// Tile index of a thread's element in the layout of a step over tile bits
// [Q, Q+RHO): element k 2^RHO + j of thread t has index ins(t + k NT) | j << Q.
template <int Q, int RHO> struct StepMap {
    static __host__ __device__ constexpr int ins(int g)
    {
        return ((g >> Q) << (Q + RHO)) | (g & ((1 << Q) - 1));
    }
    template <int NTL> static __host__ __device__ constexpr int elem(int e)
    {
        return ins((e >> RHO) << NTL) | ((e & ((1 << RHO) - 1)) << Q);
    }
};
// CKKS: lanes run over natural (not bit-reversed) positions; with K < LT the
// tile holds 2^(LT-K) blocks whose reversed block numbers are consecutive.
template <int K, int LT> struct ReverseMap {
    static __host__ __device__ constexpr int rev(int v, int bits)
    {
        int r = 0;
        for (int i = 0; i < bits; i++) r |= ((v >> i) & 1) << (bits - 1 - i);
        return r;
    }
    // whole transforms (K = n): reverse the low K bits, keep the transform
    static __host__ __device__ constexpr int whole(int g)
    {
        return ((g >> K) << K) | rev(g & ((1 << K) - 1), K);
    }
    // blocks: g = row << (LT-K) | block  ->  rev(block) << K | rev(row)
    static __host__ __device__ constexpr int blocks(int g)
    {
        return (rev(g & ((1 << (LT - K)) - 1), LT - K) << K) | rev(g >> (LT - K), K);
    }
};

// Re-deals the 16 elements of every thread: written at slots w0 ^ wc(e), read
// back from r0 ^ rc(e).  Double tiles go through 8-byte slots in two halves;
// the opaque copies of w0 and r0 keep the 32 addresses from being held in
// registers from one half to the next.  `between` (the next step's twiddle
// loads) runs once everything is written, when few registers are live.
template <typename T, typename WC, typename RC, typename B>
__device__ __forceinline__ void pass_exchange(T* lds_d, cplx<T>* v, int w0, int r0, WC wc, RC rc,
                                              bool first, B between)
{
    constexpr int EPT = 1 << PASS_E;
    if (!first) __syncthreads();
    if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int e = 0; e < EPT; e++) lds_d[w0 ^ wc(e)] = v[e].x;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EPT; e++) v[e].x = lds_d[r0 ^ rc(e)];
        __syncthreads();
        asm volatile("" : "+v"(w0));
        asm volatile("" : "+v"(r0));
#pragma unroll
        for (int e = 0; e < EPT; e++) lds_d[w0 ^ wc(e)] = v[e].y;
        between();
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EPT; e++) v[e].y = lds_d[r0 ^ rc(e)];
    } else {
        cplx<T>* lds = reinterpret_cast<cplx<T>*>(lds_d);
#pragma unroll
        for (int e = 0; e < EPT; e++) lds[w0 ^ wc(e)] = v[e];
        between();
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EPT; e++) v[e] = lds[r0 ^ rc(e)];
    }
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }

template <typename T, int MODE> __device__ __forceinline__ void butterfly(cplx<T>& U, cplx<T>& V, cplx<T> w)
{
    if constexpr (mode_is_ct(MODE)) {  // (U + V w, U - V w)
        const T xr = fma_t(-V.y, w.y, fma_t(V.x, w.x, U.x));
        const T xi = fma_t(V.y, w.x, fma_t(V.x, w.y, U.y));
        const T yr = fma_t(V.y, w.y, fma_t(-V.x, w.x, U.x));
        const T yi = fma_t(-V.y, w.x, fma_t(-V.x, w.y, U.y));
        U = mk<T>(xr, xi);
        V = mk<T>(yr, yi);
    } else {  // Gentleman-Sande: (U + V, (U - V) w)
        const cplx<T> d = U - V;
        U = U + V;
        V = d * w;
    }
}

// i sg w: a quarter turn in the table's direction (sg = +1 for a table of
// exp(+2 pi i ..), -1 for its conjugate; of the table of k-th powers, k odd: i^k)
template <typename T> __device__ __forceinline__ cplx<T> quarter(cplx<T> w, T sg)
{
    return mk<T>(-sg * w.y, sg * w.x);
}

// Twiddles of a radix-2^RHO group.  Stage ST (of the mode's order) works on
// in-group bit I with NW = 2^s distinct twiddles, in pairs a quarter turn
// apart, so only the first of each pair (the lead, u = 0 .. NW/2 - 1) is
// loaded, 8 entries per thread for 16 elements:
//   standard  s = RHO-1-I, entries (H << s) + t, H = (p >> (pb+RHO)) (+ 2^(n-pb-RHO)
//             for X^N+1), p the group's position with the step bits 0 and pb
//             the step's lowest position bit.  The tables hold bit-reversed
//             powers (fft_cpu.cu:200-211, 434-446): entry t+1 (t even) is
//             entry t times exp(sg i pi/2).
//   special   s = I, entries 2^b + (m << pb) + r, b = pb + I, r = p & (2^pb-1):
//             exp(sg 2 pi i 5^j / 2^(b+3)).  For pb >= 3, 5^(m 2^pb) = 1 - m 2^(pb+2)
//             mod 2^(pb+6), so entry m + NW/2 is entry m times exp(-sg i pi/2).
//             Steps at pb = 0 read all their entries 2^I + m (uniform).
template <int MODE, int RHO> struct Twid {
    static constexpr int bit(int st) { return mode_descending(MODE) ? RHO - 1 - st : st; }
    static constexpr int count(int st) { return 1 << (mode_special(MODE) ? bit(st) : RHO - 1 - bit(st)); }
    static constexpr int leads(int st) { return count(st) > 1 ? count(st) / 2 : 1; }
    static constexpr int first(int st)  // index of the stage's first lead
    {
        int o = 0;
        for (int i = 0; i < st; i++) o += leads(i);
        return o;
    }
};
constexpr int PASS_LEADS = 8;

// Loads leads [E0, E1) of the thread's 2^(4-RHO) groups at positions p[k].
template <typename T, int MODE, int RHO, int E0, int E1>
__device__ __forceinline__ void pass_leads(cplx<T>* lead, rsrc_t tab, int n, int nega, int pb,
                                           const int* p)
{
    using W = Twid<MODE, RHO>;
    constexpr int PER = W::first(RHO);  // leads per group
    static_assert((PER << (PASS_E - RHO)) == PASS_LEADS, "8 leads per 16 elements");
#pragma unroll
    for (int e = E0; e < E1; e++) {
        const int k = e / PER;
        int st = 0;
        for (int i = 1; i < RHO; i++)
            if (e % PER >= W::first(i)) st = i;
        const int u = e % PER - W::first(st);
        if constexpr (mode_special(MODE)) {
            lead[e] = bldc<T>(tab, (1 << (pb + W::bit(st))) + (u << pb) + (p[k] & ((1 << pb) - 1)));
        } else {
            const int H = (p[k] >> (pb + RHO)) + (nega ? 1 << (n - pb - RHO) : 0);
            lead[e] = bldc<T>(tab, (H << (RHO - 1 - W::bit(st))) + 2 * u);
        }
    }
}

// The RHO stages of one group v[0 .. 2^RHO) (v[j]: step bits = j), from stage
// ST of the mode's order on.  One twiddle at a time, so that few are live.
template <typename T, int MODE, int RHO, bool PB0, int ST = 0>
__device__ __forceinline__ void pass_group(cplx<T>* v, const cplx<T>* lead, T sg, const cplx<T>* low)
{
    if constexpr (ST < RHO) {
        using W = Twid<MODE, RHO>;
        constexpr int I = W::bit(ST);
        constexpr bool SPE = mode_special(MODE);
        constexpr int NW = W::count(ST);
        constexpr int NB = (1 << RHO) / 2 / NW;  // butterflies of each twiddle
        auto apply = [&](int t, cplx<T> w) {
#pragma unroll
            for (int x = 0; x < NB; x++) {
                const int j0 = SPE ? (x << (I + 1)) | t : (t << (I + 1)) | x;
                butterfly<T, MODE>(v[j0], v[j0 | (1 << I)], w);
            }
        };
        if constexpr (SPE && PB0) {
#pragma unroll
            for (int m = 0; m < NW; m++) apply(m, low[NW + m]);
        } else if constexpr (NW == 1) {
            apply(0, lead[W::first(ST)]);
        } else {
#pragma unroll
            for (int u = 0; u < NW / 2; u++) {
                const cplx<T> w = lead[W::first(ST) + u];
                apply(SPE ? u : 2 * u, w);
                apply(SPE ? u + NW / 2 : 2 * u + 1, quarter(w, SPE ? -sg : sg));
            }
        }
        pass_group<T, MODE, RHO, PB0, ST + 1>(v, lead, sg, low);
    }
}

// Geometry of a workgroup's tile.  Tile bits split into thread and element
// parts with no carries, so positions and offsets are sums of both parts.
template <int K, int LT, bool COL, bool REV> struct TileShape {
    static constexpr int LC = LT - K;  // log2 columns / blocks per tile
    int n, blo;
    int p0;        // position of tile element 0
    long long b0;  // its transform
    __host__ __device__ __forceinline__ void init(long long tile, int n_, int blo_)
    {
        n = n_;
        blo = blo_;
        if constexpr (COL) {
            const int ncb = blo - LC, nhi = n - blo - K;
            const int cb = (int)(tile & ((1LL << ncb) - 1));
            tile >>= ncb;
            p0 = ((int)(tile & ((1LL << nhi) - 1)) << (blo + K)) | (cb << LC);
            b0 = tile >> nhi;
        } else if (n <= LT) {
            p0 = 0;
            b0 = tile << (LT - n);
        } else {
            const int t = (int)(tile & ((1LL << (n - LT)) - 1));
            p0 = REV ? t << K : t << LT;
            b0 = tile >> (n - LT);
        }
    }
    // position (less p0) and transform (less b0) of tile index x
    __host__ __device__ __forceinline__ int pos(int x) const
    {
        if constexpr (COL) return ((x >> LC) << blo) | (x & ((1 << LC) - 1));
        if (REV && n > LT) return ((x >> K) << (n - LC)) | (x & ((1 << K) - 1));
        return n < LT ? x & ((1 << n) - 1) : x;
    }
    __host__ __device__ __forceinline__ int trn(int x) const { return (!COL && n < LT) ? x >> n : 0; }
    // element offset from transform b0, position p0
    __host__ __device__ __forceinline__ int off(int x, int stride) const { return trn(x) * stride + pos(x); }
};

// Element `lane` (thread part) of the array at `base` (uniform): a scalar base
// and a 32-bit byte offset, so that the thread part is one register for all
// its elements.
template <typename U> __device__ __forceinline__ const U& at(const U* base, int lane)
{
    return *reinterpret_cast<const U*>(reinterpret_cast<const char*>(base) +
                                       (unsigned)lane * (unsigned)sizeof(U));
}
template <typename U> __device__ __forceinline__ U& at(U* base, int lane)
{
    return *reinterpret_cast<U*>(reinterpret_cast<char*>(base) + (unsigned)lane * (unsigned)sizeof(U));
}

// Source element at (thread part xt, element part xe) of the tile.
template <typename T, int LK, typename G>
__device__ __forceinline__ cplx<T> pass_load(const RadixArgs<T>& a, const G& g, int xt, int xe)
{
    const int stride = (int)a.src_stride;
    const long long s0 = g.b0 * a.src_stride + g.p0;
    const int ot = g.off(xt, stride), oe = g.off(xe, stride);
    if constexpr (LK == LD_CPLX) {
        return at(static_cast<const cplx<T>*>(a.src) + s0 + oe, ot);
    } else if constexpr (LK == LD_REAL) {
        return mk<T>(at(static_cast<const T*>(a.src) + s0 + oe, ot), T(0));
    } else if constexpr (LK == LD_MUL) {
        const cplx<T> u = at(static_cast<const cplx<T>*>(a.src) + s0 + oe, ot);
        const cplx<T> v = at(static_cast<const cplx<T>*>(a.src2) + s0 + oe, ot);
        return u * v;
    } else if constexpr (LK == LD_FOLD) {  // (f[p] + i f[p+L]) * twist[p]
        const T* f = static_cast<const T*>(a.src) + s0 + oe;
        const cplx<T> w = at(a.ltab + g.p0 + g.pos(xe), g.pos(xt));
        return mk<T>(at(f, ot), at(f + (1 << a.n), ot)) * w;
    } else if constexpr (LK == LD_RR_PACK) {
        // Half-length form of the X^N-1 R_R inverse.  The source holds full
        // N-point spectra C in bit-reversed order (C_k at 2 bitrev(k), C_{k+M}
        // next to it, M = N/2 = 2^n); for a spectrum of real data the N-point
        // inverse D_j = sum_k C_k w^-jk has D_2m + i D_2m+1 = (M-point inverse
        // of Z)_m with Z_k = (C_k + C_{k+M}) + i w^-k (C_k - C_{k+M}), and
        // w^-k = itab[p] at bit-reversed position p = bitrev(k).  src2
        // (optional) is the second operand of the product.
        const int pt = g.pos(xt), pe = g.pos(xe);
        const long long o = (g.b0 + g.trn(xe)) * a.src_stride + 2LL * (g.p0 + pe);
        const int lane = g.trn(xt) * stride + 2 * pt;
        const cplx<T>* X = static_cast<const cplx<T>*>(a.src) + o;
        cplx<T> x0 = at(X, lane), x1 = at(X + 1, lane);
        if (a.src2) {
            const cplx<T>* Y = static_cast<const cplx<T>*>(a.src2) + o;
            x0 = x0 * at(Y, lane);
            x1 = x1 * at(Y + 1, lane);
        }
        const cplx<T> s = x0 + x1, d = (x0 - x1) * at(a.ltab + g.p0 + pe, pt);
        return mk<T>(s.x - d.y, s.y + d.x);
    } else {  // LD_SPLIT_HI / LD_SPLIT_LO: x = hi + lo, hi = float(x), lo = float(x - hi)
        const cplx<double> x = at(static_cast<const cplx<double>*>(a.src) + s0 + oe, ot);
        const T hx = (T)x.x, hy = (T)x.y;
        if constexpr (LK == LD_SPLIT_HI) return mk<T>(hx, hy);
        return mk<T>((T)(x.x - (double)hx), (T)(x.y - (double)hy));
    }
}

template <typename T, int SK, typename G>
__device__ __forceinline__ void pass_store(const RadixArgs<T>& a, const G& g, int xt, int xe, cplx<T> z)
{
    const int stride = (int)a.dst_stride;
    const long long s0 = g.b0 * a.dst_stride + g.p0;
    const int ot = g.off(xt, stride), oe = g.off(xe, stride);
    if (a.do_scale) z = z * a.scale;
    if constexpr (SK == ST_CPLX) {
        at(static_cast<cplx<T>*>(a.dst) + s0 + oe, ot) = z;
    } else if constexpr (SK == ST_REAL) {
        at(static_cast<T*>(a.dst) + s0 + oe, ot) = z.x;
    } else if constexpr (SK == ST_UNFOLD) {  // z untwist[p] -> out[p] = re, out[p+L] = im
        z = z * at(a.stab + g.p0 + g.pos(xe), g.pos(xt));
        T* o = static_cast<T*>(a.dst) + s0 + oe;
        at(o, ot) = z.x;
        at(o + (1 << a.n), ot) = z.y;
    } else {  // ST_SUM_F64: double complex dst = (double)stab[p] + (double)z
        const cplx<T> h = at(a.stab + s0 + oe, ot);
        at(static_cast<cplx<double>*>(a.dst) + s0 + oe, ot) =
            mk<double>((double)h.x + (double)z.x, (double)h.y + (double)z.y);
    }
}

// Natural coefficient index (less the tile's) of lane index x of a CKKS tile,
// and its transform; see ReverseMap.
template <int K, int LT, typename G>
__host__ __device__ __forceinline__ int ckks_index(const G& g, int x)
{
    constexpr int LC = LT - K;
    if (g.n <= LT) return (x >> K) * (2 << K) + (x & ((1 << K) - 1));
    return ((x >> LC) << (g.n - K)) | (x & ((1 << LC) - 1));
}
// First coefficient of the tile: transform b0, reversed block number.
template <int K, int LT, typename G> __device__ __forceinline__ long long ckks_base(const G& g)
{
    const long long b = g.b0 << (g.n + 1);
    if (g.n <= LT) return b;
    return b + ((__brev((unsigned)(g.p0 >> K)) >> (32 - (g.n - LT))) << (LT - K));
}

template <typename T, int MODE, int K, bool COL, int LK, int SK>
__global__ __launch_bounds__((1 << pass_tile<T>(COL, K)) >> PASS_E, 4) void radix_pass(RadixArgs<T> a)
{
    constexpr int LT = pass_tile<T>(COL, K);
    constexpr int EPT = 1 << PASS_E;
    constexpr int NTL = LT - PASS_E;  // log2 threads
    constexpr int LC = COL ? LT - K : 0;
    constexpr int NS = pass_steps(K);
    constexpr bool DESC = mode_descending(MODE);
    constexpr bool CK_IN = LK == LD_CKKS, CK_OUT = SK == ST_CKKS;
    // the global side of the step on bit 0 of a row tile goes through LDS
    constexpr bool PRE = !COL && (!DESC || NS == 1);
    constexpr bool POST = !COL && (DESC || NS == 1);
    __shared__ T lds[(sizeof(T) == 8 ? 1 : 2) << LT];

    const int tid = threadIdx.x;
    using Shape = TileShape<K, LT, COL, CK_IN || CK_OUT>;
    Shape g;
    g.init(blockIdx.x, a.n, a.blo);
    const rsrc_t tab = make_rsrc(a.tab);
    // the table's direction (Twid): tab[1] is i^k (standard), exp(k i pi/4) (special)
    T sg = T(1);
    if constexpr (K > 1) {
        const cplx<T> w1 = a.tab[1];
        if ((w1.y < T(0)) != (mode_special(MODE) && w1.x < T(0))) sg = T(-1);
    }
    // special step at bit 0: its entries are uniform, read here (ahead of any
    // barrier) so that they are scalar loads
    cplx<T> low[16];
    if constexpr (mode_special(MODE) && !COL) {
#pragma unroll
        for (int m = 1; m < (1 << pass_step_bits(K, 0)); m++) low[m] = a.tab[m];
    }

    cplx<T> v[EPT];
    bool fresh = true;  // LDS not yet used

    // step S (execution order): its first four leads, and then the others and
    // the stages
    cplx<T> lead[PASS_LEADS];
    auto leads = [&](auto step, auto half) {
        constexpr int S = decltype(step)::value;
        constexpr int as = DESC ? NS - 1 - S : S;
        constexpr int q = pass_step_q(K, as), rho = pass_step_bits(K, as);
        if constexpr (!(mode_special(MODE) && !COL && q == 0)) {
            using M = StepMap<LC + q, rho>;
            int p[EPT >> rho];
#pragma unroll
            for (int k = 0; k < (EPT >> rho); k++)
                p[k] = g.p0 + g.pos(M::ins(tid)) + g.pos(M::ins(k << NTL));
            constexpr int E0 = decltype(half)::value * (PASS_LEADS / 2);
            pass_leads<T, MODE, rho, E0, E0 + PASS_LEADS / 2>(lead, tab, a.n, a.nega,
                                                              (COL ? a.blo : 0) + q, p);
        }
    };
    auto compute = [&](auto step) {
        constexpr int S = decltype(step)::value;
        constexpr int as = DESC ? NS - 1 - S : S;
        constexpr int q = pass_step_q(K, as), rho = pass_step_bits(K, as);
        leads(step, std::integral_constant<int, 1>{});
#pragma unroll
        for (int k = 0; k < (EPT >> rho); k++)
            pass_group<T, MODE, rho, !COL && q == 0>(v + (k << rho), lead + k * (PASS_LEADS >> (PASS_E - rho)),
                                                     sg, low);
    };
    // only row tiles that hold several transforms have a tail; the full tiles'
    // accesses are unconditional (a condition around each would draw the
    // arithmetic into it)
    const bool full = COL || g.b0 + (g.n < LT ? 1 << (LT - g.n) : 1) <= a.batch;
    auto each = [&](int xt, auto elem, auto f) {
        if (full) {
#pragma unroll
            for (int e = 0; e < EPT; e++) f(e, elem(e));
        } else if constexpr (!COL) {
#pragma unroll
            for (int e = 0; e < EPT; e++)
                if (g.b0 + g.trn(xt) + g.trn(elem(e)) < a.batch) f(e, elem(e));
        }
    };
    auto zero = [&]() {
        if (!full) {
#pragma unroll
            for (int e = 0; e < EPT; e++) v[e] = mk<T>(T(0), T(0));
        }
    };
    auto linear = [](int e) { return e << NTL; };
    // loads of two or more operands go in rounds, which bounds their registers
    auto load_round = [](int e) {
        constexpr int R = LK == LD_RR_PACK ? 4 : LK == LD_MUL || LK == LD_FOLD ? 8 : EPT;
        if ((e + 1) % R == 0) __builtin_amdgcn_sched_barrier(0);
    };

    // ---- load
    zero();
    if constexpr (PRE) {
        if constexpr (CK_IN) {
            // v[bitrev(i)] = (m[i] + i m[i + l]) / delta
            const long long* m = static_cast<const long long*>(a.src) + ckks_base<K, LT>(g);
            const int it = ckks_index<K, LT>(g, tid);
            each(tid, linear, [&](int e, int x) {
                const int ie = ckks_index<K, LT>(g, x);
                v[e] = mk<T>((T)at(m + ie, it), (T)at(m + ie + (1LL << a.n), it));
            });
            if (a.inv_delta != 0.0) {  // a power of two: exact
#pragma unroll
                for (int e = 0; e < EPT; e++) v[e] = mk<T>(v[e].x * (T)a.inv_delta, v[e].y * (T)a.inv_delta);
            } else {
#pragma unroll
                for (int e = 0; e < EPT; e++) v[e] = mk<T>(v[e].x / (T)a.delta, v[e].y / (T)a.delta);
            }
        } else {
            each(tid, linear, [&](int e, int x) {
                v[e] = pass_load<T, LK>(a, g, tid, x);
                load_round(e);
            });
        }
    } else {
        constexpr int as = DESC ? NS - 1 : 0;
        using M = StepMap<LC + pass_step_q(K, as), pass_step_bits(K, as)>;
        const int xt = M::ins(tid);
        each(xt, [](int e) { return M::template elem<NTL>(e); },
             [&](int e, int x) {
                 v[e] = pass_load<T, LK>(a, g, xt, x);
                 load_round(e);
             });
    }
    auto first_leads = [&]() { leads(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}); };
    if constexpr (!PRE) first_leads();

    if constexpr (PRE) {
        using M = StepMap<pass_step_q(K, 0), pass_step_bits(K, 0)>;
        const int r0 = slot_of(M::ins(tid));
        auto rc = [](int e) { return slot_of(M::template elem<NTL>(e)); };
        if constexpr (CK_IN) {
            using R = ReverseMap<K, LT>;
            if (g.n > LT) {
                pass_exchange(lds, v, slot_of(R::blocks(tid)), r0,
                              [](int e) { return slot_of(R::blocks(e << NTL)); }, rc, fresh, first_leads);
            } else {
                pass_exchange(lds, v, slot_of(R::whole(tid)), r0,
                              [](int e) { return slot_of(R::whole(e << NTL)); }, rc, fresh, first_leads);
            }
        } else {
            pass_exchange(lds, v, slot_of(tid), r0, [](int e) { return slot_of(e << NTL); }, rc, fresh,
                          first_leads);
        }
        fresh = false;
    }
    compute(std::integral_constant<int, 0>{});

    // ---- the other steps
    auto step_on = [&](auto step) {
        constexpr int S = decltype(step)::value;
        constexpr int aw = DESC ? NS - S : S - 1, ar = DESC ? NS - 1 - S : S;
        using W = StepMap<LC + pass_step_q(K, aw), pass_step_bits(K, aw)>;
        using R = StepMap<LC + pass_step_q(K, ar), pass_step_bits(K, ar)>;
        pass_exchange(lds, v, slot_of(W::ins(tid)), slot_of(R::ins(tid)),
                      [](int e) { return slot_of(W::template elem<NTL>(e)); },
                      [](int e) { return slot_of(R::template elem<NTL>(e)); }, fresh,
                      [&]() { leads(step, std::integral_constant<int, 0>{}); });
        fresh = false;
        compute(step);
    };
    if constexpr (NS > 1) step_on(std::integral_constant<int, 1>{});
    if constexpr (NS > 2) step_on(std::integral_constant<int, 2>{});
    if constexpr (NS > 3) step_on(std::integral_constant<int, 3>{});
    static_assert(NS <= 4, "at most four radix steps");

    // ---- store
    if constexpr (POST) {
        using M = StepMap<pass_step_q(K, 0), pass_step_bits(K, 0)>;
        const int w0 = slot_of(M::ins(tid));
        auto wc = [](int e) { return slot_of(M::template elem<NTL>(e)); };
        auto nothing = []() {};
        if constexpr (CK_OUT) {
            using R = ReverseMap<K, LT>;
            if (g.n > LT) {
                pass_exchange(lds, v, w0, slot_of(R::blocks(tid)), wc,
                              [](int e) { return slot_of(R::blocks(e << NTL)); }, fresh, nothing);
            } else {
                pass_exchange(lds, v, w0, slot_of(R::whole(tid)), wc,
                              [](int e) { return slot_of(R::whole(e << NTL)); }, fresh, nothing);
            }
            // m[i] = llround(Re u[bitrev(i)] delta), m[i + l] = llround(Im ..)
            long long* m = static_cast<long long*>(a.dst) + ckks_base<K, LT>(g);
            const int it = ckks_index<K, LT>(g, tid);
            each(tid, linear, [&](int e, int x) {
                const int ie = ckks_index<K, LT>(g, x);
                const cplx<T> z = v[e] * a.scale;
                at(m + ie, it) = llround(z.x * a.delta);
                at(m + ie + (1LL << a.n), it) = llround(z.y * a.delta);
            });
        } else {
            pass_exchange(lds, v, w0, slot_of(tid), wc, [](int e) { return slot_of(e << NTL); }, fresh,
                          nothing);
            each(tid, linear, [&](int e, int x) { pass_store<T, SK>(a, g, tid, x, v[e]); });
        }
    } else {
        constexpr int as = DESC ? 0 : NS - 1;
        using M = StepMap<LC + pass_step_q(K, as), pass_step_bits(K, as)>;
        const int xt = M::ins(tid);
        each(xt, [](int e) { return M::template elem<NTL>(e); },
             [&](int e, int x) { pass_store<T, SK>(a, g, xt, x, v[e]); });
    }
}

}  // namespace gfa
