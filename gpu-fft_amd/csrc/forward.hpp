// Drop-in R_R and FFNT forward transforms of 2^13 Q double points, Q = 2^SB
// (SB = 1..3), in one launch: Q workgroups per transform, each evaluating its
// residue of the top SB stages (ForwardCore / ForwardFFNTCore order and twiddle
// indices, reference src/lib/fft.cu:11-152, 1013-1180) while it loads the whole
// transform, and the 13 stages below it in registers (subfft.hpp).  The
// workgroups of a transform run on one XCD, so its repeated reads are L2 hits;
// HBM sees every input once and every output once.
//
// The FFNT twist is part of the twiddles: the factors of positions p and
// p + 2^b differ by twist[2^b], so the stage on bit b takes root[..] twist[2^b],
// formed once per workgroup.
//
// The caller may pass the tables of the other direction.  The stages derive
// quarter turns for exp(+2 pi i ..) roots, so conjugate roots run them on
// conjugates: conj_if on the twiddles, the gathered inputs and the outputs
// (the coefficients of the gather are the table's own).
//
// Workgroups are persistent, one per CU, and load the next transform while they
// work on the current one (why, see product.hpp).  Against one workgroup per
// sub-problem with its gather, LDS steps and stores one after the other, us, on
// one buffer pair repeated and on pairs cycled beyond the last-level cache: FFNT
// N = 2^16, 512 transforms (512 MiB in and out) 132 -> 101, 152 -> 134 (4.0
// TB/s); R_R of 2^16 points x 128 61 -> 51, 61 -> 61; R_R of 2^14 points x 1024,
// read twice instead of eight times, 94 -> 64, 94 -> 66 (6.1 TB/s).  Where the
// product flow gains: persistent_forward, transform.hpp.
#pragma once

#include "oneshot.hpp"
#include "subfft.hpp"

namespace gfa {

// conj(z) if flip is the sign bit, z if it is 0
__device__ __forceinline__ cplx<double> conj_if(cplx<double> z, unsigned flip)
{
    return mk<double>(z.x, flip_sign(z.y, flip));
}

template <int SB, bool FOLD>
__global__ __launch_bounds__(512, 2) void forward13_kernel(OneArgs<double> o)
{
    constexpr int S = 13, Q = 1 << SB, NS = sub_steps(S);
    using W = Leads<S>;
    __shared__ cplx<double> lds[1 << S];
    __shared__ cplx<double> table[W::TABLE];
    const int tid = threadIdx.x;
    const int n = o.n;
    const int L = 1 << n;

    // XCD-aware order: the Q workgroups of a transform get block ids congruent mod 8
    const int slot = blockIdx.x >> 3;
    const int q = slot % Q;
    long long t = (long long)(slot / Q) * 8 + (blockIdx.x & 7);
    const long long step = gridDim.x / Q;
    const int hi = q << S;
    const double* src = static_cast<const double*>(o.src);

    // the first transform's loads, then the twiddles (a workgroup beyond the
    // last transform reads that one)
    const double* x0 = src + (t < o.batch ? t : o.batch - 1) * o.src_stride;
    GatherAll13<SB, FOLD> first;
    first.begin(x0, L, tid);

    ProdArgs<double> ra{};
    ra.n = n;
    ra.S = S;
    ra.nega = o.nega;
    ra.tab = o.tab;
    ra.twist = o.twist;
    cplx<double> C[Q];
    top_row_coeffs<double, SB, FOLD>(ra, q, C);
#pragma unroll
    for (int j = 0; j < Q; j++) C[j] = uniform(C[j]);

    // tab[1] = exp(+-i pi/2)
    const unsigned flip = o.tab[1].y < 0.0 ? 0x80000000u : 0u;
    auto entry = [&](auto qc, auto rhoc, int H, int e) {
        constexpr int lo = decltype(qc)::value, rho = decltype(rhoc)::value;
        cplx<double> w = o.tab[lead_entry<rho>(H + (o.nega ? 1 << (n - lo - rho) : 0), e)];
        if constexpr (FOLD) w = w * o.twist[1 << (lo + rho - 1 - lead_stage<rho>(e))];
        return conj_if(w, flip);
    };
    W w;
    w.table = table;
    w.load(entry, hi, tid);
#pragma unroll
    for (int e = 0; e < W::per(NS - 1); e++) w.top[e] = uniform(w.top[e]);
#pragma unroll
    for (int e = 0; e < PASS_LEADS; e++) w.mid[e] = uniform(w.mid[e]);
    static_assert(W::TABLE <= 512, "one entry per thread");
    if (tid < W::TABLE) table[tid] = w.table_entry(entry, tid, hi);

    cplx<double> v[16], next[16];
    first.end(x0, L, tid, v, C);
    arrived(v);
#pragma unroll
    for (int e = 0; e < 16; e++) v[e] = conj_if(v[e], flip);
    Gather13<SB, FOLD> gather;
    __syncthreads();
    for (; t < o.batch; t += step) {
        // (after the last one: that one's again, unused)
        const double* x = src + (t + step < o.batch ? t + step : t) * o.src_stride;
        gather.fetch(x, L, tid, 0);
        auto ahead = [&](auto I) { gather.phase(x, L, tid, next, C, decltype(I)::value); };
        sub_step<S, NS - 1, false>(v, w, tid);
        ahead(std::integral_constant<int, 0>{});
        lds_barrier();  // the tile is no longer read
        tile_write<PairMap13>(lds, v, tid);
        lds_barrier();
        tile_read<WaveMap<S, NS - 2>>(lds, v, tid);
        ahead(std::integral_constant<int, 1>{});
        sub_descend<S, NS - 2>(lds, v, w, tid, ahead);
        // consecutive lanes on consecutive outputs
        wave_fence();
        tile_write<WaveMap<S, 0>>(lds, v, tid);
        wave_fence();
        tile_read<WaveMap<S, 2>>(lds, v, tid);
        // before the stores: memory operations complete in order
        gather.finish(x, L, tid, next, C);
        arrived(next);
        cplx<double>* dst = static_cast<cplx<double>*>(o.dst) + t * o.dst_stride + hi;
#pragma unroll
        for (int e = 0; e < 16; e++)
            stc_nt(&at(dst + WaveMap<S, 2>::elem(e), WaveMap<S, 2>::ins(tid)), conj_if(v[e], flip));
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] = conj_if(next[e], flip);
    }
}

}  // namespace gfa
