// Host-side planning and launch of a full transform as a chain of passes.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "engine.hpp"
#include "oneshot.hpp"
#include "passes.hpp"
#include "product_launch.hpp"
#include "status.hpp"

namespace gfa {

struct PassPlan {
    bool col;
    int blo, K;
};

// Splits the n position bits into passes, ascending: one row pass over bits
// [0, K0) and column passes above it (pass.hpp).  One row pass up to 13 bits;
// two passes to 2^24: 8 column bits keep 128-byte column rows and two radix
// steps, and the row pass takes the rest, up to the 12 bits of the 2^12 tile;
// beyond 2^20 the column pass grows too.  (FP64, 2^23 points, batch 1, against
// 3 passes of at most 12 + 8 bits: 198 -> 100 us on one buffer, which the
// last-level cache half holds, 214 -> 136 us (3.9 TB/s) on cycled ones.)
// reversed: the CKKS passes read or write the row pass's tile in natural
// order, which needs 2^(12-K0) >= 16 blocks for 128-byte runs, so K0 <= 8.
inline std::vector<PassPlan> plan_passes(int n, bool descending, bool reversed)
{
    std::vector<PassPlan> p;
    if (n <= PASS_ROW_MAX) {
        p.push_back({false, 0, n});
        return p;
    }
    int c = n <= 16 ? n - n / 2 : n <= 20 ? 8 : n - 13 < 9 ? 9 : n - 13;
    if (reversed) c = n - 8;
    if (c <= PASS_COL_MAX) {
        p.push_back({false, 0, n - c});
        p.push_back({true, n - c, c});
    } else {
        p.push_back({false, 0, n - c});
        p.push_back({true, n - c, c / 2});
        p.push_back({true, n - c + c / 2, c - c / 2});
    }
    if (descending) std::reverse(p.begin(), p.end());
    return p;
}

// What the first pass reads and the last pass writes.
template <typename T> struct TransformIO {
    int lk;                 // LoadKind of the first pass
    const void* src;
    const void* src2;
    const cplx<T>* ltab;
    long long src_stride;
    int sk;                 // StoreKind of the last pass
    void* dst;
    const cplx<T>* stab;
    long long dst_stride;
    cplx<T>* work;          // complex [batch][2^n] buffer for intermediate passes
    bool do_scale;
    cplx<T> scale;
    double delta;           // LD_CKKS, ST_CKKS
};

// Launches every pass of one transform of length 2^n over `batch` transforms.
template <typename T>
int run_transform(int mode, int n, int batch, int nega, const cplx<T>* tab,
                  const TransformIO<T>& io, hipStream_t stream, const char* who)
{
    const bool reversed = io.lk == LD_CKKS || io.sk == ST_CKKS;
    const std::vector<PassPlan> plan = plan_passes(n, mode_descending(mode), reversed);
    const long long L = 1LL << n;
    for (size_t i = 0; i < plan.size(); i++) {
        const bool first = (i == 0), last = (i + 1 == plan.size());
        const PassPlan& pp = plan[i];
        RadixArgs<T> a{};
        a.n = n;
        a.blo = pp.blo;
        a.batch = batch;
        a.nega = nega;
        a.tab = tab;
        int lk = LD_CPLX, sk = ST_CPLX;
        if (first) {
            lk = io.lk;
            a.src = io.src;
            a.src2 = io.src2;
            a.ltab = io.ltab;
            a.src_stride = io.src_stride;
        } else {
            a.src = io.work;
            a.src_stride = L;
        }
        if (last) {
            sk = io.sk;
            a.dst = io.dst;
            a.stab = io.stab;
            a.dst_stride = io.dst_stride;
            a.do_scale = io.do_scale ? 1 : 0;
            a.scale = io.scale;
        } else {
            a.dst = io.work;
            a.dst_stride = L;
        }
        a.delta = io.delta;
        int e2 = 0;
        if (io.delta > 0 && std::frexp(io.delta, &e2) == 0.5 && std::isfinite(1.0 / io.delta))
            a.inv_delta = 1.0 / io.delta;
        RadixFn<T> fn = mode == MODE_STD_FWD ? pass_std_fwd<T>(pp.col, pp.K, lk, sk)
                      : mode == MODE_STD_INV ? pass_std_inv<T>(pp.col, pp.K, lk, sk)
                      : mode == MODE_SPE_FWD ? pass_spe_fwd<T>(pp.col, pp.K, lk, sk)
                                             : pass_spe_inv<T>(pp.col, pp.K, lk, sk);
        if (!fn) return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": no kernel for this pass");
        const int LT = pass_tile<T>(pp.col, pp.K);
        const long long tiles = (((long long)batch << n) + (1LL << LT) - 1) >> LT;
        if (tiles > 0x7fffffffLL) return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch too large");
        hipLaunchKernelGGL(fn, dim3((unsigned)tiles), dim3((1 << LT) >> PASS_E), 0, stream, a);
        GFA_CHECK_LAUNCH(who);
    }
    return ok();
}

void launch_forward13(const OneArgs<double>& a, int SB, bool fold, hipStream_t st);  // forward.hip

// Out-of-place calls (R_R, FFNT) of 2^n points, n = S + SB with S the LDS
// tile (13 double, 14 float) and SB = 1..3 (oneshot.hpp): the forward is one
// launch of Q = 2^SB workgroups per transform; the inverse is a launch of
// the in-sub-problem stages (in place in the source) and a streaming launch
// of the top SB stages with the output transform.
template <typename T> struct OneCfg;
// The forward's workgroups read the whole transform, so it takes the largest
// tile (one workgroup per CU); the inverse's first launch reads only its own
// sub-problem and takes half of it, so that two workgroups share a CU
// (measured at N = 2^16, batch 256, FP64: inverse 0.146 -> 0.135 ms; the
// forward at the smaller tile went 0.150 -> 0.161 ms).
template <> struct OneCfg<double> {
    static constexpr int S = 13, E = 4, RB = 4;   // forward: 512 threads, 16 points each
    static constexpr int SI = 12, EI = 4;         // inverse: 256 threads, 16 points each
};
template <> struct OneCfg<float> {
    static constexpr int S = 14, E = 5, RB = 4;   // forward: 512 threads, 32 points each
};

template <typename T> using OneFn = void (*)(OneArgs<T>);
template <typename T> using TopFn = void (*)(OneArgs<T>, int);

template <typename T, int SB> OneFn<T> select_forward_sb(int lk)
{
    constexpr int S = OneCfg<T>::S, E = OneCfg<T>::E, RB = OneCfg<T>::RB;
    if (lk == LD_REAL) return &fwd_sub_kernel<T, S, SB, E, RB, PL_REAL>;
    if constexpr (sizeof(T) == 8 || SB < 3) {  // the rest: prefer_passes
        if (lk == LD_FOLD) return &fwd_sub_kernel<T, S, SB, E, RB, PL_FOLD>;
    }
    return nullptr;
}

template <typename T, int SB> TopFn<T> select_top_sb(int sk)  // SB = 2..4
{
    if (sk == ST_REAL) return &inv_top_kernel<T, SB, ST_REAL>;
    if (sk == ST_UNFOLD) return &inv_top_kernel<T, SB, ST_UNFOLD>;
    return nullptr;
}

// Workgroups of a one-launch forward: transforms in groups of 8, one per XCD.
inline long long one_blocks(int batch, int SB) { return (((long long)batch + 7) / 8 * 8) << SB; }

// Where the pass chain is faster than this path (us, both sides measured, chain
// against this path):
//   FP64 forward: few transforms (the chain's workgroups are smaller): FFNT of
//     2^16 points x 2: 12.4 / 17.5, x 8 17.0 / 17.8, x 16 21.1 / 18.1; of 2^15
//     x 2 11.6 / 12.3, x 8 13.6 / 12.7; R_R of 2^16 x 2 11.6 / 12.5, x 8 15.8 /
//     12.8.  FFNT of 2^16 points has 8 workgroups to a transform, one to a CU: a
//     second wave (33 .. 64 transforms on 256 CUs) is emptier than the chain's
//     last: x 36 32.8 / 40.5, x 64 43.3 / 43.8, x 128 85 / 74.
//   FP32 inverse: R_R 2^15 x 128 17.3 / 20.7, x 1024 92 / 108; FFNT 2^15 points
//     x 256 52 / 61, x 1 10.5 / 14.0, 2^16 x 1 10.7 / 14.9.
//   FP32 forward up to 2^20 points in the launch (FFNT 2^15 x 16: 11.3 / 14.8, x
//     32 14.1 / 14.9, x 64 19.1 / 15.1; R_R 2^16 x 16 13.4 / 13.6, x 32 20 / 13.6;
//     R_R 2^15 x 16 10.5 / 12.4, x 32 13.3 / 12.6), and FFNT of 2^17 points (x 2
//     10.7 / 22.5, x 64 51 / 60).
//   FP32 forward of 2^16 and 2^17 points where the launch's second wave is at
//     most a quarter full (product flow, cycled buffers: FFNT 2^16 x 66 72 -> 64,
//     x 80 73 -> 67, R_R 2^17 x 40 66 -> 57; past that R_R 2^16 x 96 60 / 63).
// FP64 inverse, with the product (this path against the chain): R_R 2^14 x 1 9.5 /
// 10.9, x 256 56 / 66; 2^15 x 64 29 / 31; 2^16 x 1 11.6 / 11.2, x 8 15.0 / 15.1, x
// 64 57 / 66, x 512 418 / 465; FFNT 2^14 points x 1 9.9 / 12.7, x 256 62 / 72; 2^16 x
// 1 13.5 / 13.8, x 64 64 / 80, x 512 478 / 533: never the chain.
template <typename T> bool prefer_passes(bool forward, int n, int batch, bool fold, int cus)
{
    const long long points = (long long)batch << n;
    if constexpr (sizeof(T) == 8) {
        if (!forward) return false;
        if (n == 16) return batch <= (fold ? 8 : 2) || (fold && 8LL * batch > cus && 8LL * batch <= 2LL * cus);
        return n == 15 && fold && batch <= 2;
    }
    if (!forward || (n == 17 && fold)) return true;
    const long long blocks = one_blocks(batch, n - 14);
    return points <= (n == 15 && !fold ? 1LL << 19 : 1LL << 20) ||
           (n >= 16 && blocks > cus && 4 * blocks <= 5LL * cus);
}

// FP64 forwards of 2^n points in one launch: the persistent form (forward.hpp)
// instead of one workgroup per sub-problem.  It starts longer and gains from the
// second wave of workgroups on; forward and inverse with the product, repeated
// and with cycled buffers (us, per sub-problem -> persistent):
//   R_R  2^14 x 136 48 -> 46, 49 -> 46, x 256 62 -> 53, 61 -> 55; 2^15 x 72 47 -> 47, 53 -> 51,
//        x 128 62 -> 57, 64 -> 59;  2^16, eight reads of every input: x 34 50 -> 52, 57 ->
//        59, x 48 56 -> 56, 61 -> 63, x 56 61 -> 59, 65 -> 65, x 64 66 -> 63, 69 -> 67, x 72
//        86 -> 86, 93 -> 93, x 96 93 -> 92, 101 -> 98, x 128 126 -> 115, 132 -> 129
//   FFNT 2^14 points x 160 52 -> 54, 57 -> 58, x 192 56 -> 57, 61 -> 61, x 224 62 -> 61, 66 ->
//        64, x 512 144 -> 133, 151 -> 138; 2^15 x 72 54 -> 55, 63 -> 62, x 96 60 -> 58, 66 -> 66,
//        x 512 290 -> 263, 290 -> 263; 2^16 x 66 109 -> 115, 122 -> 129, x 130 182 -> 191,
//        202 -> 208, x 512 650 -> 674, 649 -> 675
inline bool persistent_forward(int n, bool fold, long long blocks, int cus)
{
    if (n == 16) return !fold && 4 * blocks >= 7LL * cus;
    return fold ? 2 * blocks >= 3LL * cus : blocks > cus;
}

// Returns true and launches when this path covers the transform (status in
// *status); false leaves the pass chain to the caller.  The source must not
// overlap the destination; the inverse uses the source as its work buffer.
template <typename T>
bool run_oneshot(int mode, int n, int batch, int nega, const cplx<T>* tab,
                 const TransformIO<T>& io, hipStream_t stream, const char* who, int* status)
{
    constexpr int S = OneCfg<T>::S, E = OneCfg<T>::E, RB = OneCfg<T>::RB;
    const int SB = n - S;
    if (SB < 1 || SB > 3) return false;
    const int cus = device_cus();
    if (prefer_passes<T>(mode == MODE_STD_FWD, n, batch, io.lk == LD_FOLD, cus)) return false;
    OneArgs<T> a{};
    a.n = n;
    a.batch = batch;
    a.nega = nega;
    a.tab = tab;
    a.twist = io.ltab;
    a.src = io.src;
    a.src2 = io.src2;
    a.src_stride = io.src_stride;
    a.dst = io.dst;
    a.dst_stride = io.dst_stride;
    a.untwist = io.stab;
    a.do_scale = io.do_scale ? 1 : 0;
    a.scale = io.do_scale ? io.scale : mk<T>(T(1), T(0));
    if (mode == MODE_STD_FWD && io.sk == ST_CPLX && (io.lk == LD_REAL || io.lk == LD_FOLD)) {
        const long long blocks = one_blocks(batch, SB);
        if (blocks > 0x7fffffffLL) {
            *status = fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch too large");
            return true;
        }
        bool launched = false;
        if constexpr (sizeof(T) == 8) {
            launched = persistent_forward(n, io.lk == LD_FOLD, blocks, cus);
            if (launched) launch_forward13(a, SB, io.lk == LD_FOLD, stream);
        }
        if (!launched) {
            OneFn<T> fn = SB == 1 ? select_forward_sb<T, 1>(io.lk)
                        : SB == 2 ? select_forward_sb<T, 2>(io.lk)
                                  : select_forward_sb<T, 3>(io.lk);
            hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3((1 << S) >> E), 0, stream, a);
        }
        hipError_t e = hipGetLastError();
        *status = e != hipSuccess ? fail_hip(e, who) : ok();
        return true;
    }
    if constexpr (sizeof(T) == 8) {
        if (mode == MODE_STD_INV && (io.lk == LD_CPLX || io.lk == LD_MUL) &&
            (io.sk == ST_REAL || io.sk == ST_UNFOLD)) {
            constexpr int SI = OneCfg<T>::SI, EI = OneCfg<T>::EI;
            const int SBI = n - SI;  // 2..4
            const long long blocks1 = (long long)batch << SBI;
            static_assert(SI >= 9, "the second inverse launch takes 512 columns per workgroup");
            const long long blocks2 = (long long)batch << (SI - 9);
            if (blocks1 > 0x7fffffffLL || blocks2 > 0x7fffffffLL) {
                *status = fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch too large");
                return true;
            }
            OneFn<T> f1 = io.lk == LD_MUL ? &inv_local_kernel<T, SI, EI, RB, LD_MUL>
                                          : &inv_local_kernel<T, SI, EI, RB, LD_CPLX>;
            hipLaunchKernelGGL(f1, dim3((unsigned)blocks1), dim3((1 << SI) >> EI), 0, stream, a);
            TopFn<T> f2 = SBI == 2 ? select_top_sb<T, 2>(io.sk)
                        : SBI == 3 ? select_top_sb<T, 3>(io.sk)
                                   : select_top_sb<T, 4>(io.sk);
            hipLaunchKernelGGL(f2, dim3((unsigned)blocks2), dim3(256), 0, stream, a, SI);
            hipError_t e = hipGetLastError();
            *status = e != hipSuccess ? fail_hip(e, who) : ok();
            return true;
        }
    }
    return false;
}

}  // namespace gfa
