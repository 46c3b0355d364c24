// Launches of the fused FP64 product kernels (product.hpp).
#include "product.hpp"

#include <algorithm>
#include <string>

#include "product_launch.hpp"
#include "status.hpp"

namespace gfa {

namespace {

using Kernel = void (*)(ProductArgs);

struct Launch {
    Kernel k, once;
    int threads, per, resident;
};

template <int S, int SB> Launch shape_of()
{
    using P = SubShape<S>;
    return {&product_kernel<S, SB, false>, &product_kernel<S, SB, true>, P::NT, P::PER, P::RESIDENT};
}

Launch select(int S, int SB)
{
    if (SB > 0 && S != 13) return {};
    switch (S) {
        case 6: return shape_of<6, 0>();
        case 7: return shape_of<7, 0>();
        case 8: return shape_of<8, 0>();
        case 9: return shape_of<9, 0>();
        case 10: return shape_of<10, 0>();
        case 11: return shape_of<11, 0>();
        case 12: return shape_of<12, 0>();
        case 13:
            switch (SB) {
                case 0: return shape_of<13, 0>();
                case 1: return shape_of<13, 1>();
                case 2: return shape_of<13, 2>();
                case 3: return shape_of<13, 3>();
                default: return {};
            }
        default: return {};
    }
}

}  // namespace

int launch_product_table(void* w, int n, int SB, hipStream_t st, const char* who)
{
    const unsigned blocks = (unsigned)((product_table_entries(n, SB) + 255) / 256);
    hipLaunchKernelGGL(product_table_kernel, dim3(blocks), dim3(256), 0, st, (cplx<double>*)w, n, SB);
    GFA_CHECK_LAUNCH(who);
    return GPUFFT_OK;
}

int launch_product_f64(int n, int S, int SB, int batch, const void* w, const double* a, const double* b,
                       double* out, void* scratch, hipStream_t st, const char* who)
{
    const Launch l = select(S, SB);
    if (!l.k) return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": no kernel for this size");
    ProductArgs pa{};
    pa.n = n;
    pa.batch = batch;
    pa.w = (const cplx<double>*)w;
    pa.a = a;
    pa.b = b;
    pa.out = out;
    pa.scratch = (cplx<double>*)scratch;
    // split products: 8 at a time, one per XCD, 2^SB workgroups each
    const long long unit = SB > 0 ? 8LL << SB : 1;
    const long long items = SB > 0 ? (((long long)batch + 7) / 8 * 8) << SB : ((long long)batch + l.per - 1) / l.per;
    const int grid = (int)std::max<long long>(unit, persistent_grid(items, l.resident) / unit * unit);
    hipLaunchKernelGGL(grid == items ? l.once : l.k, dim3((unsigned)grid), dim3(l.threads), 0, st, pa);
    GFA_CHECK_LAUNCH(who);
    return GPUFFT_OK;
}

int launch_combine_f64(int n, int S, int SB, int batch, const void* w, const void* scratch, double* out,
                       hipStream_t st, const char* who)
{
    Combine64Args ca{};
    ca.n = n;
    ca.S = S;
    ca.batch = batch;
    ca.scratch = (const cplx<double>*)scratch;
    ca.w = (const cplx<double>*)w;
    ca.out = out;
    // 512 columns per workgroup, every workgroup inside one product (S >= 9)
    const dim3 blocks((unsigned)((long long)batch << (S - 9)));
    switch (SB) {
        case 1: hipLaunchKernelGGL(combine_f64_kernel<1>, blocks, dim3(256), 0, st, ca); break;
        case 2: hipLaunchKernelGGL(combine_f64_kernel<2>, blocks, dim3(256), 0, st, ca); break;
        case 3: hipLaunchKernelGGL(combine_f64_kernel<3>, blocks, dim3(256), 0, st, ca); break;
        default: return fail(GPUFFT_ERR_UNSUPPORTED, std::string(who) + ": split too deep");
    }
    GFA_CHECK_LAUNCH(who);
    return GPUFFT_OK;
}

}  // namespace gfa
