// Launch of the one-launch double forward transforms (forward.hpp).
#include "forward.hpp"

#include <algorithm>

#include "product_launch.hpp"

namespace gfa {

void launch_forward13(const OneArgs<double>& a, int SB, bool fold, hipStream_t st)
{
    using Fn = void (*)(OneArgs<double>);
    // (FFNT of 2^16 points: never persistent, see persistent_forward)
    static constexpr Fn real[3] = {&forward13_kernel<1, false>, &forward13_kernel<2, false>,
                                   &forward13_kernel<3, false>};
    static constexpr Fn folded[2] = {&forward13_kernel<1, true>, &forward13_kernel<2, true>};
    // 8 transforms at a time, one per XCD, 2^SB workgroups each
    const long long unit = 8LL << SB;
    const long long items = (((long long)a.batch + 7) / 8 * 8) << SB;
    const Fn fn = fold ? folded[SB - 1] : real[SB - 1];
    const int grid = (int)std::max<long long>(unit, persistent_grid(items, 1) / unit * unit);
    hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(512), 0, st, a);
}

}  // namespace gfa
