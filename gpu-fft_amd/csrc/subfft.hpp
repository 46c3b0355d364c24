// Transforms of 2^S double-complex points by one workgroup, 16 points per thread
// in registers: the building blocks of the fused products (product.hpp) and
// of the one-launch forward transforms (forward.hpp).
//
// The step on the top bits works on what the operand loads deliver; one
// exchange through LDS then gives every wavefront 2^10 consecutive positions,
// and all further steps and exchanges stay inside the wavefront, without
// barriers, so wavefronts that drift apart overlap each other's LDS and
// arithmetic phases.  LDS bandwidth is the scarcest: at 2^13 points three
// exchanges per transform are 18K of its cycles per product of three transforms
// against 16K of the vector units', so one of them is done by lane swaps
// (steps of 3 | 4, 2, 4 bits; the 2-bit step takes the position bits of lane
// bits 4 and 5, which v_permlane16/32_swap trade for register bits).
#pragma once

#include "pass.hpp"

namespace gfa {

// Radix steps of a sub-problem, in ascending bit order.  2^10 and 2^13 points:
// 4, 2, 4 bits inside a wavefront's 2^10 positions (lane swaps between the
// upper two), the top 3 bits of 2^13 across wavefronts; the others as pass.hpp.
__host__ __device__ constexpr bool sub_swaps(int S) { return S == 10 || S == 13; }
__host__ __device__ constexpr int sub_steps(int S) { return S == 10 ? 3 : pass_steps(S); }
__host__ __device__ constexpr int sub_bits(int S, int s)
{
    return !sub_swaps(S) ? pass_step_bits(S, s) : s == 1 ? 2 : s == 3 ? 3 : 4;
}
__host__ __device__ constexpr int sub_q(int S, int s)
{
    return s == 0 ? 0 : sub_q(S, s - 1) + sub_bits(S, s - 1);
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
    static constexpr int NS = sub_steps(S), Q = sub_q(S, NS - 1), RHO = sub_bits(S, NS - 1);
    using M = StepMap<Q, RHO>;
    static __host__ __device__ constexpr int ins(int t) { return M::ins(t); }
    static __host__ __device__ constexpr int elem(int e) { return M::template elem<S - PASS_E>(e); }
};
// Step s of a sub-problem inside a wavefront's 2^10 positions.
template <int S, int STEP> struct WaveMap {
    using M = StepMap<sub_q(S, STEP), sub_bits(S, STEP)>;
    // the 2-bit step after the lane swaps: lane bits 5, 4 are position bits 9,
    // 8, the step's bits 5, 4 are the low element bits, bits 7, 6 the high ones
    static constexpr bool SWAPPED = sub_swaps(S) && STEP == 1;
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

// Leads are in the order of the forward stages (Twid): the stage of lead e, and
// its entry of a root table for a group at upper bits H.
template <int RHO> __device__ __forceinline__ int lead_stage(int e)
{
    int st = 0;
    for (int j = 1; j < RHO; j++)
        if (e >= Twid<MODE_STD_FWD, RHO>::first(j)) st = j;
    return st;
}
template <int RHO> __device__ __forceinline__ int lead_entry(int H, int e)
{
    const int st = lead_stage<RHO>(e);
    return (H << st) + 2 * (e - Twid<MODE_STD_FWD, RHO>::first(st));
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

// Copy of a workgroup-uniform value held in scalar registers.
__device__ __forceinline__ cplx<double> uniform(cplx<double> z)
{
    unsigned w[4];
    __builtin_memcpy(w, &z, 16);
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    __builtin_memcpy(&z, w, 16);
    return z;
}

// A wavefront's twiddles.  Steps of a sub-problem from the lowest: 0 has other
// upper bits in every thread; 1 has 2^(S-q-rho) values of them, in LDS; the top
// one (and step 2 at 2^13 points, whose upper bits are the wavefront's) has
// one.  With two steps, 1 is the top one.
template <int S> struct Leads {
    static constexpr int NS = sub_steps(S);
    static constexpr int per(int st) { return PASS_LEADS >> (PASS_E - sub_bits(S, st)); }
    static constexpr int q1 = sub_q(S, 1) + sub_bits(S, 1);
    static constexpr int TABLE = NS > 2 ? per(1) << (S - q1) : 1;  // entries of step 1 in LDS
    cplx<double> low[PASS_LEADS];
    cplx<double> mid[PASS_LEADS];  // 2^13 points: step 2
    cplx<double> top[per(NS - 1)];
    const cplx<double>* table;

    // entry(q, rho, H, e): the value of lead e of the step over bits [q, q+rho),
    // H the position bits above it; hi = the position bits above S.
    template <typename F> __device__ __forceinline__ cplx<double> table_entry(F entry, int i, int hi) const
    {
        constexpr int rho = sub_bits(S, 1);
        return entry(std::integral_constant<int, q1 - rho>{}, std::integral_constant<int, rho>{},
                     (hi >> q1) + i / per(1), i % per(1));
    }
    template <typename F> __device__ __forceinline__ void load(F entry, int hi, int tid)
    {
        constexpr int rho = sub_bits(S, 0);
        using M = WaveMap<S, 0>;
        constexpr std::integral_constant<int, 0> q0{};
        constexpr std::integral_constant<int, rho> r0{};
#pragma unroll
        for (int k = 0; k < (16 >> rho); k++) {
            const int idx = M::ins(tid) | M::elem(k << rho);
            const int p = hi | (S < 10 ? idx & ((1 << S) - 1) : idx);
#pragma unroll
            for (int e = 0; e < per(0); e++) low[k * per(0) + e] = entry(q0, r0, p >> rho, e);
        }
        constexpr int rt = sub_bits(S, NS - 1);
#pragma unroll
        for (int e = 0; e < per(NS - 1); e++)
            top[e] = entry(std::integral_constant<int, S - rt>{}, std::integral_constant<int, rt>{}, hi >> S, e);
        if constexpr (NS > 3) {
            constexpr int q2 = sub_q(S, 2), r2 = sub_bits(S, 2);
            static_assert(q2 + r2 == 10 && per(2) == PASS_LEADS, "step 2 of a 2^13-point sub-problem ends at bit 10");
            const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
            for (int e = 0; e < PASS_LEADS; e++)
                mid[e] = entry(std::integral_constant<int, q2>{}, std::integral_constant<int, r2>{},
                               (hi >> (q2 + r2)) + wave, e);
        }
    }
    // step 1's, for group k of the thread
    __device__ __forceinline__ void from_table(cplx<double>* lead, int tid, int k) const
    {
        using M = WaveMap<S, 1>;
        const int idx = M::ins(fresh(tid)) | M::elem(k << sub_bits(S, 1));
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
__device__ __forceinline__ void sub_step(cplx<double>* v, const Leads<S>& w, int tid)
{
    constexpr int rho = sub_bits(S, STEP);
    constexpr int PER = Leads<S>::per(STEP);
#pragma unroll
    for (int k = 0; k < (16 >> rho); k++) {
        cplx<double> lead[PER];
        if constexpr (STEP == 0) {
#pragma unroll
            for (int e = 0; e < PER; e++) lead[e] = w.low[k * PER + e];
        } else if constexpr (STEP == sub_steps(S) - 1) {
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
__device__ __forceinline__ void sub_move(cplx<double>* lds, cplx<double>* v, int tid)
{
    if constexpr (sub_swaps(S) && FROM + TO == 3) {
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
__device__ __forceinline__ void sub_descend(cplx<double>* lds, cplx<double>* v, const Leads<S>& w, int tid,
                                                A ahead)
{
    constexpr int I = 2 * (sub_steps(S) - 1 - STEP);
    sub_step<S, STEP, false>(v, w, tid);
    ahead(std::integral_constant<int, I>{});
    if constexpr (STEP > 0) {
        sub_move<S, STEP, STEP - 1>(lds, v, tid);
        ahead(std::integral_constant<int, I + 1>{});
        sub_descend<S, STEP - 1>(lds, v, w, tid, ahead);
    }
}
template <int S, int STEP, typename A>
__device__ __forceinline__ void sub_ascend(cplx<double>* lds, cplx<double>* v, const Leads<S>& w, int tid,
                                               A ahead)
{
    sub_step<S, STEP, true>(v, w, tid);
    ahead(std::integral_constant<int, 2 * STEP>{});
    if constexpr (STEP < sub_steps(S) - 2) {
        sub_move<S, STEP, STEP + 1>(lds, v, tid);
        ahead(std::integral_constant<int, 2 * STEP + 1>{});
        sub_ascend<S, STEP + 1>(lds, v, w, tid, ahead);
    }
}

// Workgroup shape of a 2^S-point sub-problem: 2^(S-4) threads from 2^10 points;
// below, 4 wavefronts of 2^(10-S) products each.  RESIDENT workgroups share a
// CU (2 wavefronts per SIMD at 256 registers).
template <int S> struct SubShape {
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

// Operand loads of a 2^13-point sub-problem of a transform cut into Q = 2^SB of
// them: y[c] = sum_j C[j] z_{j 2^13 + c}, C[0] = 1, in the layout PairMap13 with
// 16-byte loads, z_p = x_p + i x_{p+L} (FOLD) or x_p.  All of it at once, or, so
// that it can run ahead beside another transform, in parts: part i's rows are
// fetched by part i and added in by part i + 1.
template <int SB, bool FOLD> struct Gather13 {
    static constexpr int Q = 1 << SB;
    static constexpr int R = Q < 4 ? Q : 4;    // rows of a part
    static constexpr int PARTS = 8 * (Q / R);  // an element pair's rows take Q / R parts
    static constexpr int PPP = PARTS / 8;      // parts per phase: the start and 7 phases
    u32x4 ur[R], ui[FOLD ? R : 1];

    __device__ __forceinline__ void fetch(const double* x, int L, int tid, int i)
    {
        const rsrc_t r = make_rsrc(x);
        const int e = i / (Q / R), j0 = (i % (Q / R)) * R;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int p = ((j0 + j) << 13) | PairMap13::elem(e);
            ur[j] = __builtin_amdgcn_raw_buffer_load_b128(r, PairMap13::ins(tid) * 8, p * 8, 0);
            if constexpr (FOLD)
                ui[j] = __builtin_amdgcn_raw_buffer_load_b128(r, PairMap13::ins(tid) * 8, (p + L) * 8, 0);
        }
    }
    __device__ __forceinline__ void add_in(cplx<double>* v, const cplx<double>* C, int i)
    {
        const int e = i / (Q / R), j0 = (i % (Q / R)) * R;
#pragma unroll
        for (int j = 0; j < R; j++) {
            double re[2], im[2] = {0.0, 0.0};
            __builtin_memcpy(re, &ur[j], 16);
            if constexpr (FOLD) __builtin_memcpy(im, &ui[j], 16);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                cplx<double>& z = v[e + 8 * u];
                const cplx<double> c = C[j0 + j];
                if (j0 + j == 0) {
                    z = mk<double>(re[u], im[u]);
                } else if constexpr (FOLD) {
                    z.x = fma(-c.y, im[u], fma(c.x, re[u], z.x));
                    z.y = fma(c.y, re[u], fma(c.x, im[u], z.y));
                } else {
                    z.x = fma(c.x, re[u], z.x);
                    z.y = fma(c.y, re[u], z.y);
                }
            }
        }
    }
    // phase I (0 .. 6) of the transform beside it
    __device__ __forceinline__ void parts(const double* x, int L, int tid, cplx<double>* v, const cplx<double>* C,
                                          int i0, int i1)
    {
#pragma unroll
        for (int i = i0; i < i1; i++) {
            add_in(v, C, i - 1);
            if (i < PARTS) fetch(x, L, tid, i);
        }
    }
    __device__ __forceinline__ void phase(const double* x, int L, int tid, cplx<double>* v, const cplx<double>* C,
                                          int I)
    {
        parts(x, L, tid, v, C, I * PPP + 1, (I + 1) * PPP + 1);
    }
    // what the phases leave; everything has arrived afterwards
    __device__ __forceinline__ void finish(const double* x, int L, int tid, cplx<double>* v, const cplx<double>* C)
    {
        parts(x, L, tid, v, C, 7 * PPP + 1, 8 * PPP + 1);
    }
};
// Everything at once, up to 32 loads in flight: begin() issues the first of
// them, before what else a workgroup has to load, and end() completes v.
template <int SB, bool FOLD> struct GatherAll13 {
    using P = Gather13<SB, FOLD>;
    static constexpr int PER = P::Q / P::R;
    static constexpr int G = 32 / (P::Q * (FOLD ? 2 : 1)) < 8 ? 32 / (P::Q * (FOLD ? 2 : 1)) : 8;  // pairs in flight
    P g[G * PER];

    __device__ __forceinline__ void begin(const double* x, int L, int tid)
    {
#pragma unroll
        for (int i = 0; i < G * PER; i++) g[i].fetch(x, L, tid, i);
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void end(const double* x, int L, int tid, cplx<double>* v, const cplx<double>* C)
    {
#pragma unroll
        for (int i = 0; i < 8 * PER; i++) {
            P& s = g[i % (G * PER)];
            s.add_in(v, C, i);
            if (i + G * PER < 8 * PER) s.fetch(x, L, tid, i + G * PER);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};
__device__ __forceinline__ void arrived(cplx<double>* v)
{
#pragma unroll
    for (int e = 0; e < 16; e++) asm volatile("" : "+v"(v[e].x), "+v"(v[e].y));
}

}  // namespace gfa
