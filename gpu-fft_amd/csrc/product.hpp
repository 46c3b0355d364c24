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
// to the output stores.  The step on the top bits works on what the loads
// deliver; one exchange through LDS then gives every wavefront 2^10 consecutive
// positions, and all further steps and exchanges of the transform stay inside
// the wavefront, without barriers, so wavefronts that drift apart overlap each
// other's LDS and arithmetic phases.  LDS bandwidth is the scarcest: at 2^13
// points three exchanges per transform are 18K of its cycles per product
// against 16K of the vector units', so one of them is done by lane swaps
// (steps of 3 | 4, 2, 4 bits; the 2-bit step takes the position bits of lane
// bits 4 and 5, which v_permlane16/32_swap trade for register bits).
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
// Measured (us per call; before: one workgroup per product or sub-problem with
// every step through LDS behind barriers, a table load per twiddle stage):
//   ring 2^7  x 4096  54.5 -> 8.3     ring 2^12 x 2000  48.3 -> 40.1
//   ring 2^13 x 1     17.0 -> 12.1    ring 2^13 x 1000  60.0 -> 43.4 (4.5 TB/s)
//   ring 2^14 x 331   58.8 -> 48.7    ring 2^14 x 1000  138.7 -> 98.9 (4.0 TB/s)
//   ring 2^16 x 256   132 -> 99.6 and the combine 47 (5.7 TB/s)
// Of that, at ring 2^14 x 1000: merged twiddles, registers and wavefront-local
// exchanges 119, loads ahead 106, lane swaps 99.  At 2^13 points three LDS
// exchanges and a table load per step spilled or stalled every variant.
#pragma once

#include "pass.hpp"

namespace gfa {

struct ProductArgs {
    int n;      // log2 of the complex length L
    int batch;  // products in this launch
    const cplx<double>* w;  // merged roots W (L entries), then zeta_q^j at [L + q Q + j]
    const double* a;
    const double* b;
    double* out;            // SB = 0: [batch][2L]
    cplx<double>* scratch;  // SB > 0: [batch][L]
};

// Radix steps of a sub-problem, in ascending bit order.  2^10 and 2^13 points:
// 4, 2, 4 bits inside a wavefront's 2^10 positions (lane swaps between the
// upper two), the top 3 bits of 2^13 across wavefronts; the others as pass.hpp.
__host__ __device__ constexpr bool product_swaps(int S) { return S == 10 || S == 13; }
__host__ __device__ constexpr int product_steps(int S) { return S == 10 ? 3 : pass_steps(S); }
__host__ __device__ constexpr int product_bits(int S, int s)
{
    return !product_swaps(S) ? pass_step_bits(S, s) : s == 1 ? 2 : s == 3 ? 3 : 4;
}
__host__ __device__ constexpr int product_q(int S, int s)
{
    return s == 0 ? 0 : product_q(S, s - 1) + product_bits(S, s - 1);
}

// 16-byte LDS slot of sub-problem element i: linear over XOR, distinct banks
// for the lanes of every access below.
__host__ __device__ constexpr int slot16(int i)
{
    return i ^ ((i >> 4) & 15) ^ ((i >> 3) & 9) ^ ((i >> 2) & 14);
}

// Layout of the operand loads of a 2^13-point sub-problem: 16-byte loads bring
// two consecutive positions, so a thread holds 2 groups of the top 3 bits.
struct PairMap13 {
    static __host__ __device__ constexpr int ins(int t) { return t << 1; }
    static __host__ __device__ constexpr int elem(int e) { return (e >> 3) | ((e & 7) << 10); }
};
template <int S> struct TopMap {  // the step on the top bits, over the whole sub-problem
    static constexpr int NS = product_steps(S), Q = product_q(S, NS - 1), RHO = product_bits(S, NS - 1);
    using M = StepMap<Q, RHO>;
    static __host__ __device__ constexpr int ins(int t) { return M::ins(t); }
    static __host__ __device__ constexpr int elem(int e) { return M::template elem<S - PASS_E>(e); }
};
// Step s of a sub-problem inside a wavefront's 2^10 positions.
template <int S, int STEP> struct WaveMap {
    using M = StepMap<product_q(S, STEP), product_bits(S, STEP)>;
    // the 2-bit step after the lane swaps: lane bits 5, 4 are position bits 9,
    // 8, the step's bits 5, 4 are the low element bits, bits 7, 6 the high ones
    static constexpr bool SWAPPED = product_swaps(S) && STEP == 1;
    static __host__ __device__ constexpr int ins(int t)
    {
        if (SWAPPED) return ((t >> 6) << 10) | (((t >> 4) & 3) << 8) | (t & 15);
        return ((t >> 6) << 10) | M::ins(t & 63);
    }
    static __host__ __device__ constexpr int elem(int e)
    {
        return SWAPPED ? ((e >> 2) << 6) | ((e & 3) << 4) : M::template elem<6>(e);
    }
};

// An opaque copy of the thread index: addresses derived from it are computed
// where they are used, not kept in registers over the persistent loop.
__device__ __forceinline__ int fresh(int t)
{
    asm volatile("" : "+v"(t));
    return t;
}

template <typename W> __device__ __forceinline__ void tile_write(cplx<double>* lds, const cplx<double>* v, int tid)
{
    const int w0 = slot16(W::ins(fresh(tid)));
#pragma unroll
    for (int e = 0; e < 16; e++) lds[w0 ^ slot16(W::elem(e))] = v[e];
}
template <typename R> __device__ __forceinline__ void tile_read(const cplx<double>* lds, cplx<double>* v, int tid)
{
    const int r0 = slot16(R::ins(fresh(tid)));
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = lds[r0 ^ slot16(R::elem(e))];
}
// Orders a wavefront's LDS accesses (the hardware runs them in order).
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lead e of a group at upper bits H of a step over [q, q+rho): its entry of W
// (leads in the order of the forward stages, Twid).
template <int RHO> __device__ __forceinline__ int lead_entry(int H, int e)
{
    using W = Twid<MODE_STD_FWD, RHO>;
    int st = 0;
    for (int j = 1; j < RHO; j++)
        if (e >= W::first(j)) st = j;
    return (H << st) + 2 * (e - W::first(st));
}

// Trades lane bit LANE (4 or 5) of a pair of registers for the register bit.
template <int LANE> __device__ __forceinline__ void lane_swap(double& a, double& b)
{
    u32x2 x, y;
    __builtin_memcpy(&x, &a, 8);
    __builtin_memcpy(&y, &b, 8);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const auto r = LANE == 5 ? __builtin_amdgcn_permlane32_swap(x[i], y[i], false, false)
                                 : __builtin_amdgcn_permlane16_swap(x[i], y[i], false, false);
        x[i] = r[0];
        y[i] = r[1];
    }
    __builtin_memcpy(&a, &x, 8);
    __builtin_memcpy(&b, &y, 8);
}
// From the 4-bit step's layout (element bits 3..0 = position bits 9..6) to the
// 2-bit step's (WaveMap, SWAPPED) and back.
template <bool BACK> __device__ __forceinline__ void swap_layout(cplx<double>* v)
{
    cplx<double> u[16];
#pragma unroll
    for (int e = 0; e < 16; e++) u[e] = BACK ? v[((e & 3) << 2) | (e >> 2)] : v[e];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        lane_swap<5>(u[e].x, u[e | 8].x);
        lane_swap<5>(u[e].y, u[e | 8].y);
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
        if (e & 4) continue;
        lane_swap<4>(u[e].x, u[e | 4].x);
        lane_swap<4>(u[e].y, u[e | 4].y);
    }
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = BACK ? u[e] : u[((e & 3) << 2) | (e >> 2)];
}

// A wavefront's twiddles.  Steps of a sub-problem from the lowest: 0 has other
// upper bits in every thread; 1 has 2^(S-q-rho) values of them, in LDS; the top
// one (and step 2 at 2^13 points, whose upper bits are the wavefront's) has
// one.  With two steps, 1 is the top one.
template <int S> struct Leads {
    static constexpr int NS = product_steps(S);
    static constexpr int per(int st) { return PASS_LEADS >> (PASS_E - product_bits(S, st)); }
    static constexpr int q1 = product_q(S, 1) + product_bits(S, 1);
    static constexpr int TABLE = NS > 2 ? per(1) << (S - q1) : 1;  // entries of step 1 in LDS
    cplx<double> low[PASS_LEADS];
    cplx<double> mid[PASS_LEADS];  // 2^13 points: step 2
    cplx<double> top[per(NS - 1)];
    const cplx<double>* table;

    static __device__ __forceinline__ int table_entry(int i, int n, int hi)
    {
        const int H = (hi >> q1) + i / per(1) + (1 << (n - q1));
        return lead_entry<product_bits(S, 1)>(H, i % per(1));
    }
    __device__ __forceinline__ void load(const cplx<double>* w, int n, int hi, int tid)
    {
        constexpr int rho = product_bits(S, 0);
        using M = WaveMap<S, 0>;
        int p[16 >> rho];
#pragma unroll
        for (int k = 0; k < (16 >> rho); k++) {
            const int idx = M::ins(tid) | M::elem(k << rho);
            p[k] = hi | (S < 10 ? idx & ((1 << S) - 1) : idx);
        }
        pass_leads<double, MODE_STD_FWD, rho, 0, PASS_LEADS>(low, make_rsrc(w), n, 1, 0, p);
#pragma unroll
        for (int e = 0; e < per(NS - 1); e++)
            top[e] = w[lead_entry<product_bits(S, NS - 1)>((hi >> S) + (1 << (n - S)), e)];
        if constexpr (NS > 3) {
            constexpr int q2 = product_q(S, 2) + product_bits(S, 2);
            static_assert(q2 == 10 && per(2) == PASS_LEADS, "step 2 of a 2^13-point sub-problem ends at bit 10");
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
            for (int e = 0; e < PASS_LEADS; e++)
                mid[e] = w[lead_entry<product_bits(S, 2)>((hi >> q2) + wave + (1 << (n - q2)), e)];
        }
    }
    // step 1's, for group k of the thread
    __device__ __forceinline__ void from_table(cplx<double>* lead, int tid, int k) const
    {
        using M = WaveMap<S, 1>;
        const int idx = M::ins(fresh(tid)) | M::elem(k << product_bits(S, 1));
        const int h = (S < 10 ? idx & ((1 << S) - 1) : idx) >> q1;
#pragma unroll
        for (int e = 0; e < per(1); e++) lead[e] = table[h * per(1) + e];
    }
};

// One group's forward stages, and its inverse ones: the conjugate twiddles, the
// lowest bit first.
template <int RHO> __device__ __forceinline__ void group_fwd(cplx<double>* v, const cplx<double>* lead)
{
    pass_group<double, MODE_STD_FWD, RHO, false>(v, lead, 1.0, nullptr);
}
template <int RHO> __device__ __forceinline__ void group_inv(cplx<double>* v, const cplx<double>* lead)
{
    using F = Twid<MODE_STD_FWD, RHO>;
    using I = Twid<MODE_STD_INV, RHO>;
    cplx<double> c[PASS_LEADS >> (PASS_E - RHO)];
#pragma unroll
    for (int st = 0; st < RHO; st++)  // inverse stage st is forward stage RHO-1-st
#pragma unroll
        for (int u = 0; u < I::leads(st); u++) {
            const cplx<double> z = lead[F::first(RHO - 1 - st) + u];
            c[I::first(st) + u] = mk<double>(z.x, -z.y);
        }
    pass_group<double, MODE_STD_INV, RHO, false>(v, c, -1.0, nullptr);
}
// All groups of a thread in step STEP.
template <int S, int STEP, bool INV>
__device__ __forceinline__ void product_step(cplx<double>* v, const Leads<S>& w, int tid)
{
    constexpr int rho = product_bits(S, STEP);
    constexpr int PER = Leads<S>::per(STEP);
#pragma unroll
    for (int k = 0; k < (16 >> rho); k++) {
        cplx<double> lead[PER];
        if constexpr (STEP == 0) {
#pragma unroll
            for (int e = 0; e < PER; e++) lead[e] = w.low[k * PER + e];
        } else if constexpr (STEP == product_steps(S) - 1) {
#pragma unroll
            for (int e = 0; e < PER; e++) lead[e] = w.top[e];
        } else if constexpr (STEP == 2) {
#pragma unroll
            for (int e = 0; e < PER; e++) lead[e] = w.mid[e];
        } else {
            w.from_table(lead, tid, k);
        }
        if constexpr (INV)
            group_inv<rho>(v + (k << rho), lead);
        else
            group_fwd<rho>(v + (k << rho), lead);
    }
}

// Re-deals a wavefront's elements from the layout of step FROM to that of TO.
template <int S, int FROM, int TO>
__device__ __forceinline__ void product_move(cplx<double>* lds, cplx<double>* v, int tid)
{
    if constexpr (product_swaps(S) && FROM + TO == 3) {
        swap_layout<(TO > FROM)>(v);
    } else {
        wave_fence();
        tile_write<WaveMap<S, FROM>>(lds, v, tid);
        wave_fence();
        tile_read<WaveMap<S, TO>>(lds, v, tid);
    }
}

// Steps STEP .. 0 of the forward and STEP .. NS-2 of the inverse.  ahead(i) is
// called between the phases (part i of the loads ahead).
template <int S, int STEP, typename A>
__device__ __forceinline__ void product_descend(cplx<double>* lds, cplx<double>* v, const Leads<S>& w, int tid,
                                                A ahead)
{
    constexpr int I = 2 * (product_steps(S) - 1 - STEP);
    product_step<S, STEP, false>(v, w, tid);
    ahead(std::integral_constant<int, I>{});
    if constexpr (STEP > 0) {
        product_move<S, STEP, STEP - 1>(lds, v, tid);
        ahead(std::integral_constant<int, I + 1>{});
        product_descend<S, STEP - 1>(lds, v, w, tid, ahead);
    }
}
template <int S, int STEP, typename A>
__device__ __forceinline__ void product_ascend(cplx<double>* lds, cplx<double>* v, const Leads<S>& w, int tid,
                                               A ahead)
{
    product_step<S, STEP, true>(v, w, tid);
    ahead(std::integral_constant<int, 2 * STEP>{});
    if constexpr (STEP < product_steps(S) - 2) {
        product_move<S, STEP, STEP + 1>(lds, v, tid);
        ahead(std::integral_constant<int, 2 * STEP + 1>{});
        product_ascend<S, STEP + 1>(lds, v, w, tid, ahead);
    }
}

// Workgroup shape of a 2^S-point sub-problem: 2^(S-4) threads from 2^10 points;
// below, 4 wavefronts of 2^(10-S) products each.  RESIDENT workgroups share a
// CU (2 wavefronts per SIMD at 256 registers).
template <int S> struct ProductShape {
    static constexpr int NT = S < 10 ? 256 : 1 << (S - PASS_E);
    static constexpr int TILE = S < 10 ? 4 << 10 : 1 << S;
    static constexpr int PER = S < 10 ? 4 << (10 - S) : 1;  // products per workgroup
    static constexpr bool LOCAL = S <= 10;                  // no exchange crosses wavefronts
    static constexpr int RESIDENT = 512 / NT;
};

// Barrier of a workgroup that orders LDS only: loads ahead stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ONCE: every workgroup has one product, and nothing to load ahead for.
template <int S, int SB, bool ONCE>
__global__ __launch_bounds__(ProductShape<S>::NT, 2) void product_kernel(ProductArgs a)
{
    using P = ProductShape<S>;
    constexpr int Q = 1 << SB;
    constexpr int NS = product_steps(S);
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

    cplx<double> zeta[Q];
    if constexpr (SB > 0) {
#pragma unroll
        for (int j = 0; j < Q; j++) zeta[j] = a.w[L + q * Q + j];
    }

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
    // ---- operand loads of split products, in parts: the rows of element pair
    // e = i / (Q / R), R at a time, fetched by part i and added in by part i+1
    constexpr int R = Q < 4 ? Q : 4;      // rows of a part
    constexpr int PARTS = 8 * (Q / R);    // parts of an operand
    constexpr int PPP = PARTS / 8;        // parts per phase: the start and 7 phases (2^13 points)
    u32x4 ur[R], ui[R];
    auto fetch = [&](const double* src, long long at_p, int i) {
        const rsrc_t r = make_rsrc(src + at_p * 2 * L);
        const int e = i / (Q / R), j0 = (i % (Q / R)) * R;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int x = ((j0 + j) << S) | LoadMap::elem(e);
            ur[j] = __builtin_amdgcn_raw_buffer_load_b128(r, LoadMap::ins(tid) * 8, x * 8, 0);
            ui[j] = __builtin_amdgcn_raw_buffer_load_b128(r, LoadMap::ins(tid) * 8, (x + (int)L) * 8, 0);
        }
    };
    auto add_in = [&](cplx<double>* v, int i) {
        const int e = i / (Q / R), j0 = (i % (Q / R)) * R;
#pragma unroll
        for (int j = 0; j < R; j++) {
            double re[2], im[2];
            __builtin_memcpy(re, &ur[j], 16);
            __builtin_memcpy(im, &ui[j], 16);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                cplx<double>& z = v[e + 8 * u];
                if (j0 + j == 0) {  // zeta_q^0 = 1
                    z = mk<double>(re[u], im[u]);
                } else {
                    const cplx<double> c = zeta[j0 + j];
                    z.x = fma(-c.y, im[u], fma(c.x, re[u], z.x));
                    z.y = fma(c.y, re[u], fma(c.x, im[u], z.y));
                }
            }
        }
    };
    // the parts that phase I of the transform before takes, and the last ones
    auto parts = [&](const double* src, long long at_p, cplx<double>* v, int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; i++) {
            add_in(v, i - 1);
            if (i < PARTS) fetch(src, at_p, i);
        }
    };
    // the last parts; the loads have arrived afterwards
    auto finish = [&](const double* src, long long at_p, cplx<double>* v) {
        if constexpr (SB > 0) parts(src, at_p, v, 7 * PPP + 1, 8 * PPP + 1);
#pragma unroll
        for (int e = 0; e < 16; e++) asm volatile("" : "+v"(v[e].x), "+v"(v[e].y));
    };
    // everything (SB = 0) or part 0
    auto start = [&](const double* src, long long at_p, cplx<double>* v) {
        if constexpr (SB > 0)
            fetch(src, at_p, 0);
        else
            load(src, at_p, v);
    };

    // forward transform of v (in LoadMap), to the layout of step 0
    W w;
    w.table = table;
    auto forward = [&](cplx<double>* v, auto ahead) {
        product_step<S, NS - 1, false>(v, w, tid);
        ahead(std::integral_constant<int, 0>{});
        if constexpr (P::LOCAL) {
            product_move<S, NS - 1, NS - 2>(lds, v, tid);
        } else {
            lds_barrier();  // the tile is no longer read
            tile_write<LoadMap>(lds, v, tid);
            lds_barrier();
            tile_read<WaveMap<S, NS - 2>>(lds, v, tid);
        }
        ahead(std::integral_constant<int, 1>{});
        product_descend<S, NS - 2>(lds, v, w, tid, ahead);
    };

    w.load(a.w, n, hi, tid);
    constexpr int LR = (W::TABLE + P::NT - 1) / P::NT;
    cplx<double> entry[LR];
    if constexpr (NS > 2) {
#pragma unroll
        for (int i = 0; i < LR; i++)
            entry[i] = a.w[W::table_entry((tid + i * P::NT) % W::TABLE, n, hi)];
    }
    cplx<double> vb[16], va[16];
    if ((AHEAD || ONCE) && p < a.batch) start(a.b, p, vb);
    if (ONCE && !PAIR && p < a.batch) start(a.a, p, va);
    if constexpr (NS > 2) {
#pragma unroll
        for (int i = 0; i < LR; i++)
            if (tid + i * P::NT < W::TABLE) table[tid + i * P::NT] = entry[i];
    }
    if ((AHEAD || (ONCE && PAIR)) && p < a.batch) {
        if constexpr (SB > 0) parts(a.b, p, vb, 1, 7 * PPP + 1);
        finish(a.b, p, vb);
    }
    __syncthreads();
    for (; p < a.batch; p += ONCE ? a.batch : step) {
        if constexpr (!AHEAD && !ONCE) start(a.b, p, vb);
        if constexpr (!ONCE || PAIR) start(a.a, p, va);
        forward(vb, [&](auto phase) {
            constexpr int I = decltype(phase)::value;
            if constexpr (SB > 0) parts(a.a, p, va, I * PPP + 1, (I + 1) * PPP + 1);
        });
        if constexpr (AHEAD || PAIR) finish(a.a, p, va);
        forward(va, [](auto) {});
#pragma unroll
        for (int e = 0; e < 16; e++) va[e] = va[e] * vb[e];
        // (after the last product: that one's again, unused; a condition around
        // the loads costs registers)
        const long long next = p + step < a.batch ? p + step : p;
        if constexpr (AHEAD) start(a.b, next, vb);
        auto ahead = [&](auto phase) {
            constexpr int I = decltype(phase)::value;
            if constexpr (SB > 0 && AHEAD) parts(a.b, next, vb, I * PPP + 1, (I + 1) * PPP + 1);
        };
        product_ascend<S, 0>(lds, va, w, tid, ahead);
        if constexpr (P::LOCAL) {
            product_move<S, NS - 2, NS - 1>(lds, va, tid);
        } else {
            wave_fence();
            tile_write<WaveMap<S, NS - 2>>(lds, va, tid);
            lds_barrier();
            tile_read<StoreMap>(lds, va, tid);
        }
        ahead(std::integral_constant<int, 2 * NS - 3>{});
        product_step<S, NS - 1, true>(va, w, tid);
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

// Fills W (2^n entries) and the residue powers zeta_q^j (2^SB x 2^SB) behind it.
__global__ void product_table_kernel(cplx<double>* w, int n, int SB)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    const int L = 1 << n, Q = 1 << SB;
    if (k >= L + Q * Q) return;
    // angle 2 pi num / den, exact
    double num = 0.0, den = 1.0;
    if (k >= L) {
        const int q = (k - L) >> SB, j = (k - L) & (Q - 1);
        const int r = SB ? (int)(__brev((unsigned)q) >> (32 - SB)) : 0;
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
