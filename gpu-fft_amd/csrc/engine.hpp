// Radix steps through LDS, shared by the fused products, the batched kernel and
// the one-launch drop-in transforms: a workgroup holds a sub-problem of 2^K
// points in LDS (XOR-swizzled in 16-element blocks against bank conflicts) and
// runs radix-2^RHO steps on it, each thread taking groups of 2^RHO points to
// registers and back.  Modes and load/store kinds are shared with the pass
// kernels (pass.hpp, where the stage semantics are described).
#pragma once

#include "cplx.hpp"

namespace gfa {

enum Mode { MODE_STD_FWD = 0, MODE_STD_INV = 1, MODE_SPE_FWD = 2, MODE_SPE_INV = 3 };
enum LoadKind {
    LD_CPLX = 0,
    LD_REAL = 1,
    LD_MUL = 2,
    LD_FOLD = 3,
    LD_SPLIT_HI = 4,  // T = float: double complex source, its float rounding
    LD_SPLIT_LO = 5,  // T = float: double complex source, the float of the rest
    LD_RR_PACK = 6,   // R_R inverse by half-length packing (see pass_load)
    LD_CKKS = 7,      // T = double: int64 coefficients / delta, bit-reversed positions
};
enum StoreKind {
    ST_CPLX = 0,
    ST_REAL = 1,
    ST_UNFOLD = 2,
    ST_SUM_F64 = 3,  // T = float: double complex dst = (double)aux[p] + (double)z
    ST_CKKS = 4,     // T = double: llround(z delta) to int64 coefficients, bit-reversed positions
};

__host__ __device__ constexpr bool mode_is_ct(int m) { return m == MODE_STD_FWD || m == MODE_SPE_FWD; }
__host__ __device__ constexpr bool mode_descending(int m) { return m == MODE_STD_FWD || m == MODE_SPE_INV; }
__host__ __device__ constexpr bool mode_special(int m) { return m == MODE_SPE_FWD || m == MODE_SPE_INV; }

template <typename T> struct PassArgs {
    int n;       // log2 transform length
    int K;       // number of bits (stages) of the sub-problem
    int nega;    // X^N+1 twiddle base (standard modes only)
    const cplx<T>* tab;  // root-of-unity table (reference layout)
    unsigned conj;       // TW (group_stages_derived): the sign bit if tab[1] = -i, 0 if it is i
};

// Bank-conflict swizzle: permutes each aligned block of 16 elements by the
// XOR of the next two 4-bit fields of the index.
__device__ __forceinline__ int swz(int i) { return i ^ (((i >> 4) ^ (i >> 8)) & 15); }

// Position (within its transform) of tile row r, column col.
struct TileGeo {
    int hi_pos;   // (hi << (blo+K)) | c0
    int blo, K, logC;
    rsrc_t tab;   // root-of-unity table
    __device__ __forceinline__ int pos(int r, int col) const
    {
        return hi_pos | ((r & ((1 << K) - 1)) << blo) | col;
    }
};

template <typename T, int MODE>
__device__ __forceinline__ int twiddle_index(int n, int nega, int b, int p)
{
    if constexpr (mode_special(MODE)) {
        return (1 << b) + (p & ((1 << b) - 1));
    } else {
        int base = nega ? (1 << (n - 1 - b)) : 0;
        return base + (p >> (b + 1));
    }
}

// Standard-mode stages with derived twiddles.  Inside a step over bits
// [q, q+RHO) every twiddle of the stage with in-group bit i is
//     table[base + ((P >> (q+RHO)) << s) + t] = table[base + ((P >> (q+RHO)) << s)]
//                                             * exp(2 pi i bitrev_s(t) / 2^(s+1)),
// s = RHO-1-i, t < 2^s the group bits above i (the reference tables hold
// bit-reversed powers, fft_cpu.cu:200-211 and 434-446, so an index t below
// a multiple of 2^s only adds a root of order 2^(s+1)).  One table load per
// stage; wc[2^s + t] holds the root constants (s < 5), or, with TW, the
// root table itself does at wc[t]: every reference table (FFT<T>, FFNT<T>,
// forward or inverse, either reduction) has tab[t] = exp(+-2 pi i bitrev_s(t)
// / 2^(s+1)) for t < 2^s.  The values differ from direct table reads by
// rounding only.
template <typename T, int MODE, int RHO, bool TW = false>
__device__ __forceinline__ void group_stages_derived(cplx<T>* v, const PassArgs<T>& a,
                                                     const TileGeo& g, int rbase, int col, int q,
                                                     const cplx<T>* __restrict__ wc)
{
    static_assert(!mode_special(MODE), "derived twiddles are for the standard modes");
#pragma unroll
    for (int st = 0; st < RHO; st++) {
        const int i = mode_descending(MODE) ? (RHO - 1 - st) : st;
        const int s = RHO - 1 - i;
        const int bpos = g.blo + q + i;
        const int p0 = g.pos(rbase, col);
        const cplx<T> base = bldc<T>(g.tab, twiddle_index<T, MODE>(a.n, a.nega, bpos, p0));
#pragma unroll
        for (int t = 0; t < (1 << s); t++) {
            cplx<T> w = base;
            if (TW && t == 1 && s == 1) {
                // times tab[1] = exp(+-i pi/2), exact
                w = mk<T>(flip_sign(base.y, a.conj ^ 0x80000000u), flip_sign(base.x, a.conj));
            } else if (t == 1 && s == 1) {
                // the same of the plans' own tables: forward chains use the
                // roots, inverse chains (Gentleman-Sande) their conjugates
                w = mode_is_ct(MODE) ? mk<T>(-base.y, base.x) : mk<T>(base.y, -base.x);
            } else if (t > 0) {
                w = base * wc[TW ? t : (1 << s) + t];
            }
#pragma unroll
            for (int lo = 0; lo < (1 << i); lo++) {
                const int j0 = (t << (i + 1)) | lo;
                const int j1 = j0 | (1 << i);
                cplx<T> U = v[j0], V = v[j1];
                if constexpr (mode_is_ct(MODE)) {
                    cplx<T> Vw = V * w;
                    v[j0] = U + Vw;
                    v[j1] = U - Vw;
                } else {
                    v[j0] = U + V;
                    v[j1] = (U - V) * w;
                }
            }
        }
    }
}

// Group geometry of thread `tid`, k-th group, for a step over tile-row bits
// [q, q+RHO): the group's rows are rbase | (j << q).
template <int RHO, int NT>
__device__ __forceinline__ void group_of(int tid, int k, int logC, int q, int& rbase, int& col)
{
    const int gamma = tid + k * NT;
    col = gamma & ((1 << logC) - 1);
    const int rest = gamma >> logC;
    const int rlo = rest & ((1 << q) - 1);
    const int rhi = rest >> q;
    rbase = (rhi << (q + RHO)) | rlo;
}

// One radix-2^RHO step over tile-row bits [q, q+RHO): every thread takes
// EPT/2^RHO groups of 2^RHO elements from LDS, runs the RHO stages in
// registers and writes them back.
template <typename T, int MODE, int E, int RHO, int NT, bool TW = false>
__device__ __forceinline__ void radix_step(cplx<T>* lds, const PassArgs<T>& a, const TileGeo& g,
                                           int q, int tid, const cplx<T>* wc = nullptr)
{
    constexpr int GS = 1 << RHO;
    constexpr int GPT = (1 << E) / GS;
    // the groups of a thread are processed one after the other: the fused
    // kernels are tight on registers
#pragma unroll 1
    for (int k = 0; k < GPT; k++) {
        int rbase, col;
        group_of<RHO, NT>(tid, k, g.logC, q, rbase, col);
        cplx<T> v[GS];
#pragma unroll
        for (int j = 0; j < GS; j++) v[j] = lds[swz(((rbase | (j << q)) << g.logC) | col)];
        group_stages_derived<T, MODE, RHO, TW>(v, a, g, rbase, col, q, wc);
#pragma unroll
        for (int j = 0; j < GS; j++) lds[swz(((rbase | (j << q)) << g.logC) | col)] = v[j];
    }
}

// Steps [S, SEND) of a pass of K bits with radix-2^RB steps, unrolled at
// compile time so that every step's bit range is a constant (address and
// twiddle-index arithmetic then folds).
template <typename T, int MODE, int E, int NT, int K, int RB, int S, int SEND, bool TW = false>
__device__ __forceinline__ void run_steps_ct(cplx<T>* lds, const PassArgs<T>& a, const TileGeo& g,
                                             int tid, const cplx<T>* wc)
{
    if constexpr (S < SEND) {
        constexpr int full = K / RB;
        constexpr int rem = K - full * RB;
        constexpr int nst = full + (rem ? 1 : 0);
        constexpr int as = mode_descending(MODE) ? (nst - 1 - S) : S;
        constexpr int q = as * RB;
        constexpr int rho = (as < full) ? RB : rem;
        __syncthreads();
        radix_step<T, MODE, E, rho, NT, TW>(lds, a, g, q, tid, wc);
        run_steps_ct<T, MODE, E, NT, K, RB, S + 1, SEND, TW>(lds, a, g, tid, wc);
    } else {
        __syncthreads();
    }
}

// run_steps_ct for workgroups larger than the tile's thread count: every
// thread takes the barriers, only the first NT threads compute.
template <typename T, int MODE, int E, int NT, int K, int RB, int S, int SEND>
__device__ __forceinline__ void run_steps_ct_active(cplx<T>* lds, const PassArgs<T>& a,
                                                    const TileGeo& g, int tid, const cplx<T>* wc,
                                                    bool active)
{
    if constexpr (S < SEND) {
        constexpr int full = K / RB;
        constexpr int rem = K - full * RB;
        constexpr int nst = full + (rem ? 1 : 0);
        constexpr int as = mode_descending(MODE) ? (nst - 1 - S) : S;
        constexpr int q = as * RB;
        constexpr int rho = (as < full) ? RB : rem;
        __syncthreads();
        if (active) radix_step<T, MODE, E, rho, NT>(lds, a, g, q, tid, wc);
        run_steps_ct_active<T, MODE, E, NT, K, RB, S + 1, SEND>(lds, a, g, tid, wc, active);
    } else {
        __syncthreads();
    }
}

}  // namespace gfa
