// Fused batched polynomial multiplication (additive API; the reference needs
// two GPU_FFNT calls and a caller-side rounding for the same product,
// example/test_ffnt_gpu_R_R.cu:137-162).
//
// A plan owns its root tables (generated on the GPU in FP64: the merged roots
// of product.hpp, or the reference's FFNT layouts for the FP32 split) and the
// scratch buffer of the split kernels.
//   GPUFFT_PREC_F64        double in, double out (unrounded, like GPU_FFNT)
//   GPUFFT_PREC_F32_SPLIT  int32 in, int64 out: the operands are split into
//                          balanced base-2^w limbs, every limb product runs in
//                          FP32 and is rounded, and the rounded limb products
//                          are recombined exactly in int64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "fused.hpp"
#include "product_launch.hpp"
#include "status.hpp"

using namespace gfa;

struct gpufft_polymul_plan_s {
    int device;
    int ring_power;  // log2 N
    int n;           // log2 L, L = N/2
    int precision;
    int max_batch;
    int wa, ka, wb, kb;
    int ca;          // FP32 split: a split as a - 2^ca (0: none), plus the limb 2^ca J b
    void* jspec;     // FP32 split with ca: forward FFNT spectrum of J (complex float, L)
    int S, SB;       // sub-problem split
    int rb;          // FP32 split: radix bits per LDS step of the product kernel
    int e;           // FP32 split: log2 points per thread of the product kernel (2^(S-e) threads)
    int cmb;         // FP64, SB > 0: 1 = PHASE_TRANSFORM runs the combine too
    void* root;      // FP64: merged roots (product.hpp); FP32 split: forward FFNT root table (L entries)
    void* iroot;
    void* twist;
    void* untwist;
    void* wc;        // stage root constants and their conjugates (32 each)
    void* wci;
    void* scratch;
    size_t scratch_bytes;
};

namespace {

constexpr int F64_MAX_S = 13;  // 2^13 doubles complex = 128 KiB of LDS
constexpr int F32_MAX_S = 14;  // 2^14 floats complex = 128 KiB of LDS
constexpr int MAX_SB = 3;
constexpr int F64_E = 4;   // FP64 plans: log2 points per thread

using ProdKernel = void (*)(ProdArgs<float>);

// Zero fill by a kernel rather than hipMemsetAsync, so that a caller may
// capture the call into a HIP graph.
__global__ void zero_kernel(double* p, long long n)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

__global__ void fill_ones(float* p, long long n)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 1.0f;
}

// Whether the product kernel exists for a sub-problem of 2^S points, 2^E
// points per thread and radix-2^RB steps: the thread's groups of V loaded
// positions must hold the 2^(S mod RB) partners of the register top step.
template <int S, int E, int RB> constexpr bool prod_ok()
{
    constexpr int HB = S % RB;
    constexpr int V = in_vec<float, PL_FOLD_LIMB, E, HB>();
    return RB <= E && S > E && ((1 << E) / V) / (1 << HB) >= 1;
}

// FP32 split, 2^E points per thread: 2^(S-E) threads per workgroup
template <int RB, int E> ProdKernel prod_kernel_rb(int S, int SB)
{
#define GFA_PK(SS, BB)                                                 \
    if constexpr (prod_ok<SS, E, RB>())                                \
        if (S == SS && SB == BB) return &product_sub_kernel<SS, BB, E, RB>;
    GFA_PK(7, 0)
    GFA_PK(8, 0)
    GFA_PK(9, 0)
    GFA_PK(10, 0)
    GFA_PK(11, 0)
    GFA_PK(12, 0)
    GFA_PK(13, 0)
    GFA_PK(14, 0)
    GFA_PK(14, 1)
    GFA_PK(14, 2)
    GFA_PK(14, 3)
#undef GFA_PK
    return nullptr;
}

// radix bits per LDS step 3..5, points per thread 2^e: 32 or 16; both chosen
// per plan
template <int E> ProdKernel prod_kernel_e(int S, int SB, int rb)
{
    switch (rb) {
        case 3: return prod_kernel_rb<3, E>(S, SB);
        case 4: return prod_kernel_rb<4, E>(S, SB);
        case 5:
            if constexpr (E >= 5) return prod_kernel_rb<5, E>(S, SB);
            return nullptr;
        default: return nullptr;
    }
}

ProdKernel prod_kernel(int S, int SB, int rb, int e)
{
    if (e == 5) return prod_kernel_e<5>(S, SB, rb);
    if (e == 4) return prod_kernel_e<4>(S, SB, rb);
    return nullptr;
}

int make_f64_table(gpufft_polymul_plan_s* pl, hipStream_t st)
{
    hipError_t e = hipMalloc(&pl->root, sizeof(cplx<double>) * product_table_entries(pl->n, pl->SB));
    if (e != hipSuccess) return fail_hip(e, "gpufft_polymul_plan_create: hipMalloc");
    return launch_product_table(pl->root, pl->n, pl->SB, st, "gpufft_polymul_plan_create");
}

int make_f32_tables(gpufft_polymul_plan_s* pl, hipStream_t st)
{
    size_t bytes = sizeof(cplx<float>) << pl->n;
    void** dst[4] = {&pl->root, &pl->iroot, &pl->twist, &pl->untwist};
    for (void** d : dst) {
        hipError_t e = hipMalloc(d, bytes);
        if (e != hipSuccess) return fail_hip(e, "gpufft_polymul_plan_create: hipMalloc");
    }
    for (void** d : {&pl->wc, &pl->wci}) {
        hipError_t e = hipMalloc(d, sizeof(cplx<float>) * 32);
        if (e != hipSuccess) return fail_hip(e, "gpufft_polymul_plan_create: hipMalloc");
    }
    int s;
    if ((s = gpufft_generate_table_f32(pl->root, GPUFFT_TABLE_FFNT_ROOT, pl->n, 0, st))) return s;
    if ((s = gpufft_generate_table_f32(pl->iroot, GPUFFT_TABLE_FFNT_ROOT, pl->n, 1, st))) return s;
    if ((s = gpufft_generate_table_f32(pl->twist, GPUFFT_TABLE_FFNT_TWIST, pl->n, 0, st))) return s;
    if ((s = gpufft_generate_table_f32(pl->untwist, GPUFFT_TABLE_FFNT_TWIST, pl->n, 1, st))) return s;
    if ((s = gpufft_generate_table_f32(pl->wc, GPUFFT_TABLE_STAGE_ROOTS, 5, 0, st))) return s;
    if ((s = gpufft_generate_table_f32(pl->wci, GPUFFT_TABLE_STAGE_ROOTS, 5, 1, st))) return s;
    return GPUFFT_OK;
}

void release(gpufft_polymul_plan_s* pl)
{
    if (!pl) return;
    void* ptrs[8] = {pl->root, pl->iroot, pl->twist, pl->untwist, pl->wc, pl->wci, pl->scratch,
                     pl->jspec};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    delete pl;
}

// FP32-split transforms and limb products into the plan's scratch
int launch_split(const gpufft_polymul_plan_s* pl, const int32_t* a, const int32_t* b, int batch,
                 hipStream_t st, const char* who)
{
    ProdArgs<float> pa{};
    pa.n = pl->n;
    pa.S = pl->S;
    pa.batch = batch;
    pa.nega = 0;
    pa.tab = (const cplx<float>*)pl->root;
    pa.itab = (const cplx<float>*)pl->iroot;
    pa.twist = (const cplx<float>*)pl->twist;
    pa.untwist = (const cplx<float>*)pl->untwist;
    pa.wc = (const cplx<float>*)pl->wc;
    pa.wci = (const cplx<float>*)pl->wci;
    pa.a = a;
    pa.b = b;
    pa.in_stride = 2LL << pl->n;
    pa.scratch = (cplx<float>*)pl->scratch;
    pa.wa = pl->wa;
    pa.ka = pl->ka;
    pa.ca = pl->ca;
    pa.jspec = (const cplx<float>*)pl->jspec;
    pa.wb = pl->wb;
    pa.kb = pl->kb;
    auto offset = [](int w, int k) {
        long long o = 0;
        for (int j = 0; j + 1 < k; j++) o += (1LL << (w - 1)) << (w * j);
        return o;
    };
    pa.oa = pl->ka > 1 ? offset(pl->wa, pl->ka) : 0;
    pa.ob = pl->kb > 1 ? offset(pl->wb, pl->kb) : 0;
    ProdKernel k = prod_kernel(pl->S, pl->SB, pl->rb, pl->e);
    if (!k) return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": no kernel for this size");
    const int threads = (1 << pl->S) >> pl->e;
    const long long groups = ((long long)batch + 7) / 8;
    const long long blocks = groups * 8 * (1LL << pl->SB);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(threads), 0, st, pa);
    GFA_CHECK_LAUNCH(who);
    return GPUFFT_OK;
}

int check_plan(const gpufft_polymul_plan_s* pl, int precision, int batch, const char* who)
{
    if (!pl) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": plan is NULL");
    if (pl->precision != precision)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": plan precision mismatch");
    if (batch < 1) return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch must be >= 1");
    return GPUFFT_OK;
}

// FP64 products of a validated plan (or of the no-allocation entry point's
// stack plan), in launches of at most max_batch products.
int run_f64(const gpufft_polymul_plan_s* plan, const double* a, const double* b, double* out,
            int batch, int phases, hipStream_t st, const char* who)
{
    const long long N = 2LL << plan->n;
    const int S = plan->S, SB = plan->SB;
    const bool transform = phases & GPUFFT_PHASE_TRANSFORM;
    // combine_in_kernel: PHASE_TRANSFORM writes the output, PHASE_COMBINE
    // alone does nothing
    const bool combine = SB > 0 && (plan->cmb ? transform : (phases & GPUFFT_PHASE_COMBINE) != 0);
    for (int b0 = 0; b0 < batch; b0 += plan->max_batch) {
        const int nb = std::min(plan->max_batch, batch - b0);
        if (transform)
            if (int s = launch_product_f64(plan->n, S, SB, nb, plan->root, a + b0 * N, b + b0 * N,
                                           out + b0 * N, plan->scratch, st, who))
                return s;
        if (combine)
            if (int s = launch_combine_f64(plan->n, S, SB, nb, plan->root, plan->scratch, out + b0 * N,
                                           st, who))
                return s;
    }
    return ok();
}

// ---- products without allocation ----
// Static device scratch of gpufft_polymul_f64_noalloc: the merged root tables
// (every call writes its ring's) and the sub-problem results of products split
// over several workgroups (64 MiB).  Each device holds its own copy from module
// load until the process ends.  No entry of a table depends on which ring's call
// wrote it: unsplit rings take the first roots of the longest table, and the
// split ones, whose residue powers stand behind the roots, have a table each.
// So calls that overlap in time on one device race for the sub-problem results
// only (split rings).
// First entry of the split table of 2^n points (n = 13: the end of them all).
constexpr size_t noalloc_table(int n)
{
    size_t at = 0;
    for (int k = F64_MAX_S + MAX_SB; k > n; k--) at += product_table_entries(k, k - F64_MAX_S);
    return at;
}
constexpr size_t NOALLOC_TABLE_BYTES = (sizeof(cplx<double>) * noalloc_table(F64_MAX_S) + 4095) / 4096 * 4096;
constexpr size_t NOALLOC_BYTES = NOALLOC_TABLE_BYTES + ((size_t)64 << 20);
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex noalloc_mu;
void* noalloc_ptr[NOALLOC_MAX_DEVICES];  // device address of `scratch`, per device

// Device address of this device's `scratch`, looked up once per device with
// the device current (the host-side name is only a stand-in).
int noalloc_scratch(int dev, void** out, const char* who)
{
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
        return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": device index out of range");
    std::lock_guard<std::mutex> lock(noalloc_mu);
    if (!noalloc_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            return fail_hip(e != hipSuccess ? e : hipErrorInvalidSymbol, who);
        }
        noalloc_ptr[dev] = p;
    }
    *out = noalloc_ptr[dev];
    return GPUFFT_OK;
}

}  // namespace

extern "C" {

int gpufft_polymul_plan_create(gpufft_polymul_plan* out, int ring_power, int precision,
                               int max_batch, int a_limb_bits, int a_limbs, int b_limb_bits,
                               int b_limbs, void* stream)
{
    const char* who = "gpufft_polymul_plan_create";
    if (!out) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": out is NULL");
    *out = nullptr;
    if (precision != GPUFFT_PREC_F64 && precision != GPUFFT_PREC_F32_SPLIT)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": unknown precision");
    const int E = precision == GPUFFT_PREC_F64 ? 4 : 5;
    const int smax = precision == GPUFFT_PREC_F64 ? F64_MAX_S : F32_MAX_S;
    const int n = ring_power - 1;
    if (n < E + 2 || n > smax + MAX_SB)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT,
                    std::string(who) + ": ring_power out of the fused range");
    if (max_batch < 1) return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": max_batch < 1");
    if (precision == GPUFFT_PREC_F32_SPLIT) {
        if (a_limbs < 1 || b_limbs < 1 || a_limbs * b_limbs > 64 ||
            (a_limbs > 1 && (a_limb_bits < 1 || a_limb_bits > 16)) ||
            (b_limbs > 1 && (b_limb_bits < 1 || b_limb_bits > 16)) ||
            (a_limbs > 1 && (a_limbs - 1) * a_limb_bits > 30) ||
            (b_limbs > 1 && (b_limbs - 1) * b_limb_bits > 30))
            return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": invalid limb split");
    }
    gpufft_polymul_plan_s* pl = new gpufft_polymul_plan_s();
    (void)hipGetDevice(&pl->device);
    pl->ring_power = ring_power;
    pl->n = n;
    pl->precision = precision;
    pl->max_batch = max_batch;
    if (precision == GPUFFT_PREC_F32_SPLIT) {
        pl->wa = a_limbs > 1 ? a_limb_bits : 0;
        pl->ka = a_limbs;
        pl->wb = b_limbs > 1 ? b_limb_bits : 0;
        pl->kb = b_limbs;
    } else {
        pl->ka = pl->kb = 1;
    }
    pl->S = std::min(n, smax);
    pl->SB = n - pl->S;
    pl->rb = 4;
    // FP32: 1024 threads of 16 points per full 2^14-point tile (measured
    // faster than 512 threads of 32 at N = 2^16: 0.38 against 0.45 ms per
    // batch of 256), 512 threads of 32 points below the full tile
    // FP32: 16 points per thread (1024 threads) for full tiles of products
    // in one or two sub-problems; with more, the top-row gather's partner
    // loads spill at 128 VGPRs and 32 points per thread (256 VGPRs) is faster
    pl->e = precision == GPUFFT_PREC_F64 ? F64_E : (pl->S == F32_MAX_S && pl->SB <= 1 ? 4 : 5);
    pl->cmb = 0;
    hipStream_t st = (hipStream_t)stream;
    int s = precision == GPUFFT_PREC_F64 ? make_f64_table(pl, st) : make_f32_tables(pl, st);
    if (s) {
        release(pl);
        return s;
    }
    const bool need_scratch = precision == GPUFFT_PREC_F32_SPLIT || pl->SB > 0;
    if (need_scratch) {
        size_t elem = precision == GPUFFT_PREC_F64 ? 16 : 8;
        // FP32 split: room for the optional J limb (gpufft_polymul_plan_set_a_center)
        const size_t limbs = precision == GPUFFT_PREC_F32_SPLIT ? (size_t)(pl->ka + 1) * pl->kb : 1;
        pl->scratch_bytes = (size_t)max_batch * limbs * (elem << n);
        hipError_t e = hipMalloc(&pl->scratch, pl->scratch_bytes);
        if (e != hipSuccess) {
            release(pl);
            return fail_hip(e, "gpufft_polymul_plan_create: hipMalloc scratch");
        }
    }
    // tables are ready before the plan is used on any stream
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        release(pl);
        return fail_hip(e, "gpufft_polymul_plan_create: table generation");
    }
    *out = pl;
    return ok();
}

int gpufft_polymul_plan_destroy(gpufft_polymul_plan plan)
{
    release(plan);
    return GPUFFT_OK;
}

int gpufft_polymul_f64(gpufft_polymul_plan plan, const double* a, const double* b, double* out,
                       int batch, void* stream)
{
    return gpufft_polymul_f64_phases(plan, a, b, out, batch, GPUFFT_PHASE_ALL, stream);
}

int gpufft_polymul_f64_phases(gpufft_polymul_plan plan, const double* a, const double* b,
                              double* out, int batch, int phases, void* stream)
{
    const char* who = "gpufft_polymul_f64";
    if (int s = check_plan(plan, GPUFFT_PREC_F64, batch, who)) return s;
    if (!a || !b || !out) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": NULL buffer");
    return run_f64(plan, a, b, out, batch, phases, (hipStream_t)stream, who);
}

int gpufft_polymul_i32(gpufft_polymul_plan plan, const int32_t* a, const int32_t* b, int64_t* out,
                       int batch, double* err_stats, void* stream)
{
    return gpufft_polymul_i32_phases(plan, a, b, out, batch, err_stats, GPUFFT_PHASE_ALL, stream);
}

int gpufft_polymul_i32_phases(gpufft_polymul_plan plan, const int32_t* a, const int32_t* b,
                              int64_t* out, int batch, double* err_stats, int phases, void* stream)
{
    const char* who = "gpufft_polymul_i32";
    if (int s = check_plan(plan, GPUFFT_PREC_F32_SPLIT, batch, who)) return s;
    if (!a || !b || !out) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": NULL buffer");
    hipStream_t st = (hipStream_t)stream;
    const long long N = 2LL << plan->n;
    if (err_stats && (phases & GPUFFT_PHASE_COMBINE)) {
        const long long cnt = 2LL * batch;
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, st,
                           err_stats, cnt);
        GFA_CHECK_LAUNCH(who);
    }
    for (int b0 = 0; b0 < batch; b0 += plan->max_batch) {
        const int nb = std::min(plan->max_batch, batch - b0);
        if (phases & GPUFFT_PHASE_TRANSFORM)
            if (int s = launch_split(plan, a + b0 * N, b + b0 * N, nb, st, who))
                return s;
        if (!(phases & GPUFFT_PHASE_COMBINE)) continue;
        const long long nthreads_total = (long long)nb << plan->S;
        if ((nthreads_total + 255) / 256 > 0x7fffffffLL)
            return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch too large");
        const unsigned blocks = (unsigned)((nthreads_total + 255) / 256);
#define GFA_COMB(BB)                                                                       \
    case BB: {                                                                             \
        CombineArgs<BB> ca{};                                                              \
        ca.n = plan->n;                                                                    \
        ca.S = plan->S;                                                                    \
        ca.batch = nb;                                                                     \
        ca.nprod = (plan->ka + (plan->ca ? 1 : 0)) * plan->kb;                             \
        ca.ka = plan->ka;                                                                  \
        ca.ca = plan->ca;                                                                  \
        ca.kb = plan->kb;                                                                  \
        ca.wa = plan->wa;                                                                  \
        ca.wb = plan->wb;                                                                  \
        ca.scratch = (const cplx<float>*)plan->scratch;                                    \
        ca.itab = (const cplx<float>*)plan->iroot;                                         \
        ca.untwist = (const cplx<float>*)plan->untwist;                                    \
        ca.scale = (float)(1.0 / (double)(1LL << plan->n));                                \
        ca.out = (long long*)(out + b0 * N);                                               \
        ca.out_stride = N;                                                                 \
        ca.err = err_stats ? err_stats + 2 * b0 : nullptr;                                 \
        hipLaunchKernelGGL(limb_combine_kernel<BB>, dim3(blocks), dim3(256), 0, st, ca);   \
        break;                                                                             \
    }
        switch (plan->SB) {
            GFA_COMB(0)
            GFA_COMB(1)
            GFA_COMB(2)
            GFA_COMB(3)
            default: return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": split too deep");
        }
#undef GFA_COMB
        GFA_CHECK_LAUNCH(who);
    }
    return ok();
}

size_t gpufft_polymul_plan_scratch_bytes(gpufft_polymul_plan plan)
{
    return plan ? plan->scratch_bytes : 0;
}

int gpufft_polymul_plan_set_radix_bits(gpufft_polymul_plan plan, int radix_bits)
{
    const char* who = "gpufft_polymul_plan_set_radix_bits";
    if (!plan) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": plan is NULL");
    const int hi = plan->precision == GPUFFT_PREC_F64 ? 4 : 5;
    if (radix_bits < 3 || radix_bits > hi)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": radix_bits out of range");
    if (plan->precision == GPUFFT_PREC_F32_SPLIT &&
        !prod_kernel(plan->S, plan->SB, radix_bits, plan->e))
        return fail(GPUFFT_ERR_UNSUPPORTED,
                    std::string(who) + ": no kernel for this radix at the plan's points per thread");
    plan->rb = radix_bits;
    return ok();
}

int gpufft_polymul_plan_set_thread_points(gpufft_polymul_plan plan, int log2_points)
{
    const char* who = "gpufft_polymul_plan_set_thread_points";
    if (!plan) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": plan is NULL");
    const bool okv = plan->precision == GPUFFT_PREC_F64 ? log2_points == F64_E
                                                        : (log2_points == 4 || log2_points == 5);
    if (!okv) return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": unsupported points per thread");
    if (plan->precision == GPUFFT_PREC_F32_SPLIT &&
        !prod_kernel(plan->S, plan->SB, plan->rb, log2_points))
        return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": no kernel for this size and radix");
    plan->e = log2_points;
    return ok();
}

int gpufft_polymul_plan_get_thread_points(gpufft_polymul_plan plan)
{
    return plan ? plan->e : -1;
}

int gpufft_polymul_plan_get_radix_bits(gpufft_polymul_plan plan)
{
    return plan ? plan->rb : -1;
}

int gpufft_polymul_plan_set_combine(gpufft_polymul_plan plan, int in_kernel)
{
    const char* who = "gpufft_polymul_plan_set_combine";
    if (!plan) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": plan is NULL");
    if (in_kernel != 0 && in_kernel != 1)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": in_kernel must be 0 or 1");
    // only FP64 plans with more than one workgroup per product have the choice
    plan->cmb = plan->precision == GPUFFT_PREC_F64 && plan->SB > 0 ? in_kernel : 0;
    return ok();
}

int gpufft_polymul_plan_get_combine(gpufft_polymul_plan plan)
{
    return plan ? plan->cmb : -1;
}

int gpufft_polymul_plan_set_a_center(gpufft_polymul_plan plan, int center_log2)
{
    const char* who = "gpufft_polymul_plan_set_a_center";
    if (!plan) return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": plan is NULL");
    if (plan->precision != GPUFFT_PREC_F32_SPLIT)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": only GPUFFT_PREC_F32_SPLIT plans");
    if (center_log2 < 0 || center_log2 > 30)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": center_log2 must be 0..30");
    if (center_log2 > 0 && !plan->jspec) {
        // spectrum of J (all ones), once per plan: the GPU_FFNT forward of the
        // plan's own tables, so it is the transform the product kernel applies
        const long long N = 2LL << plan->n, L = 1LL << plan->n;
        hipError_t e = hipMalloc(&plan->jspec, sizeof(cplx<float>) * (size_t)L);
        if (e != hipSuccess) return fail_hip(e, "gpufft_polymul_plan_set_a_center: hipMalloc");
        float* ones = nullptr;
        e = hipMalloc((void**)&ones, sizeof(float) * (size_t)N);
        if (e != hipSuccess) {
            (void)hipFree(plan->jspec);
            plan->jspec = nullptr;
            return fail_hip(e, "gpufft_polymul_plan_set_a_center: hipMalloc");
        }
        hipLaunchKernelGGL(fill_ones, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, 0, ones, N);
        gpufft_config cfg{};
        cfg.n_power = plan->ring_power;
        cfg.fft_type = GPUFFT_FORWARD;
        cfg.stream = nullptr;
        int st = gpufft_ffnt_f32(ones, plan->jspec, plan->twist, plan->root, &cfg, 1, 0);
        hipError_t e2 = hipDeviceSynchronize();
        (void)hipFree(ones);
        if (st) return st;
        if (e2 != hipSuccess) return fail_hip(e2, "gpufft_polymul_plan_set_a_center: J spectrum");
    }
    plan->ca = center_log2;
    return ok();
}

int gpufft_polymul_plan_get_a_center(gpufft_polymul_plan plan)
{
    return plan ? plan->ca : -1;
}

int gpufft_polymul_f64_noalloc(const double* a, const double* b, double* out, int ring_power,
                               int batch, const void* twist, const void* untwist,
                               const void* root_table, const void* inv_root_table, void* stream)
{
    const char* who = "gpufft_polymul_f64_noalloc";
    const int n = ring_power - 1;
    if (n < 4 + 2 || n > F64_MAX_S + MAX_SB)
        return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": ring_power must be 7..17");
    if (batch < 1) return fail(GPUFFT_ERR_INVALID_ARGUMENT, std::string(who) + ": batch must be >= 1");
    if (!a || !b || !out || !twist || !untwist || !root_table || !inv_root_table)
        return fail(GPUFFT_ERR_NULL_POINTER, std::string(who) + ": NULL buffer");
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail_hip(e, who);
    void* base = nullptr;
    if (int s = noalloc_scratch(dev, &base, who)) return s;
    hipStream_t st = (hipStream_t)stream;
    gpufft_polymul_plan_s pl{};
    pl.device = dev;
    pl.ring_power = ring_power;
    pl.n = n;
    pl.precision = GPUFFT_PREC_F64;
    pl.ka = pl.kb = 1;
    pl.S = std::min(n, F64_MAX_S);
    pl.SB = n - pl.S;
    pl.root = (cplx<double>*)base + (pl.SB > 0 ? noalloc_table(n) : 0);
    // the sub-problem results of one launch must fit the rest of the array:
    // the batch runs in launches of at most that many products
    const size_t per_product = pl.SB > 0 ? (sizeof(cplx<double>) << n) : 0;
    const size_t room = NOALLOC_BYTES - NOALLOC_TABLE_BYTES;
    pl.max_batch = per_product ? (int)std::min<size_t>(room / per_product, (size_t)batch) : batch;
    pl.scratch = pl.SB > 0 ? (void*)((unsigned char*)base + NOALLOC_TABLE_BYTES) : nullptr;
    pl.scratch_bytes = pl.SB > 0 ? room : 0;
    // the merged roots: written by every call (a kernel, so the call can be
    // captured into a graph), ahead of the product kernels on `st`
    if (int s = launch_product_table(pl.root, n, pl.SB, st, who)) return s;
    return run_f64(&pl, a, b, out, batch, GPUFFT_PHASE_ALL, st, who);
}

}  // extern "C"
