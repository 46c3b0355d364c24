// Fused FP64 polynomial products mod X^N + 1 for gfx950.
//
// A product folds its operands to L = N/2 = 2^n complex points z_p = x_p + i x_{p+L},
// transforms both mod X^L - i, multiplies pointwise and transforms back.  With the
// roots of X^L = i instead of twist + cyclic transform (the reference's GPU_FFNT,
// src/lib/fft.cu:1013-1384) the twist is part of the twiddles: the stage on position
// bit b, upper bits h, has twiddle W[2^s + h], s = n-1-b,
//     W[2^s + t] = exp(2 pi i (1/4 + bitrev_s(t)) / 2^(s+1)),
// which is root[h] twist[2^b] of the reference's tables (the twist factors of
// positions p and p + 2^b differ by twist[2^b]); spectra and products are the same
// up to rounding, and the inverse uses the conjugates.
//
// Up to 2^13 points a product is one workgroup (or, below 2^10 points, several
// products one wavefront).  Longer ones are cut into Q = 2^SB sub-problems of
// 2^13 points, one workgroup each: residues mod X^(2^S) - zeta_q, zeta_q =
// exp(2 pi i (1/4 + bitrev_SB(q)) / Q), evaluated while loading,
//     y_q[c] = sum_j zeta_q^j z_{j 2^S + c}
// (the Q workgroups of a product run on one XCD, close in time, so the repeated
// operand reads are L2 hits), and combine_f64_kernel runs the top SB inverse
// stages from the sub-results in scratch.
//
// A thread holds 16 points of each operand in registers from the operand loads
// to the output stores (subfft.hpp).
//
// At 2^13 points one workgroup fills a CU (128 KiB of LDS, 8 wavefronts of up
// to 256 registers), so nothing else would hide its memory phases (37 us of
// loads and 28 us of stores in 119 us for 1000 products of ring 2^14, all CUs
// loading, computing and storing in step).  Hence the workgroups are
// persistent and load ahead: operand a while b is transformed, the next
// product's b during the inverse (split products a part at each stage, as
// their 2^SB rows do not fit the registers).  Loads return in order, so
// nothing else may load from memory meanwhile: a wavefront keeps its twiddles
// for life, those of the lowest step in vector registers, the uniform ones of
// the top steps in scalar registers, and the rest in a small LDS table.
//
// Measured (us per call on one set of buffers repeated, and on sets cycled
// beyond the last-level cache; before: one workgroup per product or sub-problem
// with every step through LDS behind barriers, a table load per twiddle stage):
//   ring 2^7  x 4096  54.8 -> 8.3, 57.9 -> 9.4     ring 2^12 x 2000  50 -> 42, 60 -> 48
//   ring 2^13 x 1     17.1 -> 12.1, 19.4 -> 12.4   ring 2^13 x 1000  62 -> 44, 73 -> 53 (3.7 TB/s)
//   ring 2^14 x 331   59 -> 49, 65 -> 54           ring 2^14 x 1000  141 -> 100, 139 -> 100 (3.9 TB/s)
//   ring 2^16 x 256   133 -> 103, 156 -> 122, and the combine 44 (6.1 TB/s)
// Of that, at ring 2^14 x 1000: merged twiddles, registers and wavefront-local
// exchanges 119, loads ahead 106, lane swaps 99.  At 2^13 points three LDS
// exchanges and a table load per step spilled or stalled every variant.
#pragma once

#include "subfft.hpp"

namespace gfa {

struct ProductArgs {
    int n;      // log2 of the complex length L
    int batch;  // products in this launch
    const cplx<double>* w;  // merged roots W (L entries), for SB > 0 then zeta_q^j at [L + q Q + j]
    const double* a;
    const double* b;
    double* out;            // SB = 0: [batch][2L]
    cplx<double>* scratch;  // SB > 0: [batch][L]
};

// ONCE: every workgroup has one product, and nothing to load ahead for.
template <int S, int SB, bool ONCE>
__global__ __launch_bounds__(SubShape<S>::NT, 2) void product_kernel(ProductArgs a)
{
    using P = SubShape<S>;
    constexpr int Q = 1 << SB;
    constexpr int NS = sub_steps(S);
    constexpr bool PAIR = S == 13;   // 16-byte operand loads
    // b is loaded ahead in the round before, else at the start of the round
    constexpr bool AHEAD = S >= 10 && !ONCE;
    static_assert(SB == 0 || PAIR, "split products are cut into 2^13-point sub-problems");
    using W = Leads<S>;
    __shared__ cplx<double> lds[P::TILE];
    __shared__ cplx<double> table[W::TABLE];
    const int tid = threadIdx.x;
    const int n = a.n;
    const long long L = 1LL << n;

    // The workgroup's products: p, p + step, ...  Split ones: consecutive
    // workgroups go to consecutive XCDs, so the Q workgroups of one product
    // get block ids congruent mod 8.
    int q = 0;
    long long p = (long long)blockIdx.x * P::PER, step = (long long)gridDim.x * P::PER;
    if constexpr (SB > 0) {
        const int x = blockIdx.x, slot = x >> 3;
        q = slot % Q;
        p = (long long)(slot / Q) * 8 + (x & 7);
        step = gridDim.x / Q;
    }
    const int hi = q << S;

    // layouts of the operand loads and of the output stores
    using LoadMap = std::conditional_t<PAIR, PairMap13, std::conditional_t<P::LOCAL, WaveMap<S, NS - 1>, TopMap<S>>>;
    using StoreMap = std::conditional_t<P::LOCAL, WaveMap<S, NS - 1>, TopMap<S>>;
    // element offset of tile index x, a sum over its thread and element parts
    auto off = [](int x) { return S < 10 ? ((x >> S) * (2 << S)) | (x & ((1 << S) - 1)) : x; };

    // ---- operand loads, whole (SB = 0) ----
    auto load = [&](const double* src, long long at_p, cplx<double>* v) {
        const double* x = src + at_p * 2 * L;
        const int xt = off(LoadMap::ins(tid));
        if constexpr (PAIR) {
            const rsrc_t r = make_rsrc(x);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                double re[2], im[2];
                const u32x4 ur = __builtin_amdgcn_raw_buffer_load_b128(r, xt * 8, LoadMap::elem(e) * 8, 0);
                const u32x4 ui = __builtin_amdgcn_raw_buffer_load_b128(r, xt * 8, (LoadMap::elem(e) + (int)L) * 8, 0);
                __builtin_memcpy(re, &ur, 16);
                __builtin_memcpy(im, &ui, 16);
                v[e] = mk<double>(re[0], im[0]);
                v[e + 8] = mk<double>(re[1], im[1]);
            }
        } else if (at_p + P::PER <= a.batch) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const double* y = x + off(LoadMap::elem(e));
                v[e] = mk<double>(at(y, xt), at(y + L, xt));
            }
        } else {  // the last products: those beyond the batch read its last one
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int i = LoadMap::ins(tid) | LoadMap::elem(e);
                const long long pr = at_p + (i >> S) < a.batch ? at_p + (i >> S) : a.batch - 1;
                const double* y = src + pr * 2 * L + (i & ((1 << S) - 1));
                v[e] = mk<double>(y[0], y[L]);
            }
        }
    };
    // b of the first product, ahead of the twiddles (a workgroup beyond the
    // last product reads that one)
    const double* b0 = a.b + (p < a.batch ? p : a.batch - 1) * 2 * L;
    GatherAll13<SB, true> first;
    if constexpr (SB > 0) first.begin(b0, (int)L, tid);

    cplx<double> zeta[Q];  // zeta_q^j
    if constexpr (SB > 0) {
#pragma unroll
        for (int j = 0; j < Q; j++) zeta[j] = a.w[L + q * Q + j];
    }
    // split products: in parts, beside another transform (Gather13)
    Gather13<SB, true> gather;
    auto phase = [&](const double* src, long long at_p, cplx<double>* v, int I) {
        if constexpr (SB > 0) gather.phase(src + at_p * 2 * L, (int)L, tid, v, zeta, I);
    };
    auto finish = [&](const double* src, long long at_p, cplx<double>* v) {
        if constexpr (SB > 0) gather.finish(src + at_p * 2 * L, (int)L, tid, v, zeta);
        arrived(v);
    };
    // everything (SB = 0) or part 0
    auto start = [&](const double* src, long long at_p, cplx<double>* v) {
        if constexpr (SB > 0)
            gather.fetch(src + at_p * 2 * L, (int)L, tid, 0);
        else
            load(src, at_p, v);
    };

    // forward transform of v (in LoadMap), to the layout of step 0
    W w;
    w.table = table;
    auto forward = [&](cplx<double>* v, auto ahead) {
        sub_step<S, NS - 1, false>(v, w, tid);
        ahead(std::integral_constant<int, 0>{});
        if constexpr (P::LOCAL) {
            sub_move<S, NS - 1, NS - 2>(lds, v, tid);
        } else {
            lds_barrier();  // the tile is no longer read
            tile_write<LoadMap>(lds, v, tid);
            lds_barrier();
            tile_read<WaveMap<S, NS - 2>>(lds, v, tid);
        }
        ahead(std::integral_constant<int, 1>{});
        sub_descend<S, NS - 2>(lds, v, w, tid, ahead);
    };

    auto entry = [&](auto qc, auto rhoc, int H, int e) {
        constexpr int top = decltype(qc)::value + decltype(rhoc)::value;
        return a.w[lead_entry<decltype(rhoc)::value>(H + (1 << (n - top)), e)];
    };
    w.load(entry, hi, tid);
    constexpr int LR = (W::TABLE + P::NT - 1) / P::NT;
    cplx<double> slot[LR];
    if constexpr (NS > 2) {
#pragma unroll
        for (int i = 0; i < LR; i++)
            slot[i] = w.table_entry(entry, (tid + i * P::NT) % W::TABLE, hi);
    }
    cplx<double> vb[16], va[16];
    if constexpr (SB == 0) {
        if ((AHEAD || ONCE) && p < a.batch) start(a.b, p, vb);
        if (ONCE && !PAIR && p < a.batch) start(a.a, p, va);
    }
    if constexpr (NS > 2) {
#pragma unroll
        for (int i = 0; i < LR; i++)
            if (tid + i * P::NT < W::TABLE) table[tid + i * P::NT] = slot[i];
    }
    if constexpr (SB > 0) first.end(b0, (int)L, tid, vb, zeta);
    if ((AHEAD || (ONCE && PAIR)) && p < a.batch) arrived(vb);
    __syncthreads();
    for (; p < a.batch; p += ONCE ? a.batch : step) {
        if constexpr (!AHEAD && !ONCE) start(a.b, p, vb);
        if constexpr (!ONCE || PAIR) start(a.a, p, va);
        forward(vb, [&](auto I) { phase(a.a, p, va, decltype(I)::value); });
        if constexpr (AHEAD || PAIR) finish(a.a, p, va);
        forward(va, [](auto) {});
#pragma unroll
        for (int e = 0; e < 16; e++) va[e] = va[e] * vb[e];
        // (after the last product: that one's again, unused; a condition around
        // the loads costs registers)
        const long long next = p + step < a.batch ? p + step : p;
        if constexpr (AHEAD) start(a.b, next, vb);
        auto ahead = [&](auto I) {
            if constexpr (AHEAD) phase(a.b, next, vb, decltype(I)::value);
        };
        sub_ascend<S, 0>(lds, va, w, tid, ahead);
        if constexpr (P::LOCAL) {
            sub_move<S, NS - 2, NS - 1>(lds, va, tid);
        } else {
            wave_fence();
            tile_write<WaveMap<S, NS - 2>>(lds, va, tid);
            lds_barrier();
            tile_read<StoreMap>(lds, va, tid);
        }
        ahead(std::integral_constant<int, 2 * NS - 3>{});
        sub_step<S, NS - 1, true>(va, w, tid);
        ahead(std::integral_constant<int, 2 * NS - 2>{});
        // before the stores: memory operations complete in order, so b would
        // wait for them in the next round
        if constexpr (AHEAD) finish(a.b, next, vb);

        if constexpr (SB > 0) {
            cplx<double>* dst = a.scratch + p * L + hi;
#pragma unroll
            for (int e = 0; e < 16; e++) stc_nt(&at(dst + StoreMap::elem(e), StoreMap::ins(tid)), va[e]);
        } else {
            const double scale = 1.0 / (double)(1 << S);
            double* o = a.out + p * 2 * L;
            if (p + P::PER <= a.batch) {
                const int xt = off(StoreMap::ins(tid));
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    double* y = o + off(StoreMap::elem(e));
                    at(y, xt) = va[e].x * scale;
                    at(y + L, xt) = va[e].y * scale;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int i = StoreMap::ins(tid) | StoreMap::elem(e);
                    if (p + (i >> S) < a.batch) {
                        o[off(i)] = va[e].x * scale;
                        o[off(i) + L] = va[e].y * scale;
                    }
                }
            }
        }
    }
}

// The top SB inverse stages (bits S .. n-1) of split products, the scale and
// the unfold: out[P] = Re, out[P + L] = Im.  A workgroup takes 512 consecutive
// columns of one product, each thread the columns c and c + 256: the lanes of
// every load read consecutive 16-byte scratch entries and the lanes of every
// store write consecutive doubles.
struct Combine64Args {
    int n, S, batch;
    const cplx<double>* scratch;  // [batch][2^n]
    const cplx<double>* w;
    double* out;                  // [batch][2 2^n]
};

template <int SB> __global__ __launch_bounds__(256) void combine_f64_kernel(Combine64Args a)
{
    constexpr int Q = 1 << SB;
    const long long g0 = (long long)blockIdx.x * 512;
    const long long p = g0 >> a.S;
    const int c = (int)(g0 & ((1LL << a.S) - 1)) + threadIdx.x;
    if (p >= a.batch) return;
    const long long L = 1LL << a.n;
    const cplx<double>* src = a.scratch + p * L;
    cplx<double> y[2][Q];
#pragma unroll
    for (int j = 0; j < Q; j++) {
        y[0][j] = ldc_nt(src + ((long long)j << a.S) + c);
        y[1][j] = ldc_nt(src + ((long long)j << a.S) + c + 256);
    }
#pragma unroll
    for (int i = 0; i < SB; i++) {
#pragma unroll
        for (int j0 = 0; j0 < Q; j0++) {
            if (j0 & (1 << i)) continue;
            const int j1 = j0 | (1 << i);
            const cplx<double> t = a.w[(1 << (SB - 1 - i)) + (j0 >> (i + 1))];
#pragma unroll
            for (int v = 0; v < 2; v++)
                butterfly<double, MODE_STD_INV>(y[v][j0], y[v][j1], mk<double>(t.x, -t.y));
        }
    }
    const double scale = 1.0 / (double)L;
    double* o = a.out + p * 2 * L;
#pragma unroll
    for (int j = 0; j < Q; j++) {
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const int P = (j << a.S) | (c + 256 * v);
            __builtin_nontemporal_store(y[v][j].x * scale, o + P);
            __builtin_nontemporal_store(y[v][j].y * scale, o + P + L);
        }
    }
}

// Fills W (2^n entries, the first ones of every longer W) and, for SB > 0, the
// residue powers zeta_q^j (2^SB x 2^SB) behind it.
__global__ void product_table_kernel(cplx<double>* w, int n, int SB)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    const int L = 1 << n, Q = 1 << SB;
    if (k >= L + (SB > 0 ? Q * Q : 0)) return;
    // angle 2 pi num / den, exact
    double num = 0.0, den = 1.0;
    if (k >= L) {
        const int q = (k - L) >> SB, j = (k - L) & (Q - 1);
        const int r = (int)(__brev((unsigned)q) >> (32 - SB));
        num = (double)((1 + 4 * r) * j);
        den = 4.0 * Q;
    } else if (k > 0) {
        const int s = 31 - __clz(k);
        const int r = s ? (int)(__brev((unsigned)(k - (1 << s))) >> (32 - s)) : 0;
        num = 1.0 + 4.0 * r;
        den = 8.0 * (1 << s);
    }
    double sn, cs;
    sincospi(2.0 * num / den, &sn, &cs);
    w[k] = mk<double>(cs, sn);
}

}  // namespace gfa
