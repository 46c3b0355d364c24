// Lookup of the radix pass kernels (pass.hpp); one translation unit per
// element type and mode holds their code.
#pragma once

#include "pass.hpp"

namespace gfa {

template <typename T> using RadixFn = void (*)(RadixArgs<T>);

constexpr int PASS_ROW_MAX = 13;  // row passes take 1 .. 13 bits
constexpr int PASS_COL_MIN = 6;   // column passes 6 .. 11
constexpr int PASS_COL_MAX = 11;

// Kernel of a pass over K bits; nullptr for what no operation uses.
template <typename T> RadixFn<T> pass_std_fwd(bool col, int K, int lk, int sk);
template <typename T> RadixFn<T> pass_std_inv(bool col, int K, int lk, int sk);
template <typename T> RadixFn<T> pass_spe_fwd(bool col, int K, int lk, int sk);
template <typename T> RadixFn<T> pass_spe_inv(bool col, int K, int lk, int sk);

template <typename T, int MODE, bool COL, int LK, int SK, int K0, int K1> RadixFn<T> pass_pick(int K)
{
    if constexpr (K0 > K1)
        return nullptr;
    else
        return K == K0 ? &radix_pass<T, MODE, K0, COL, LK, SK>
                       : pass_pick<T, MODE, COL, LK, SK, K0 + 1, K1>(K);
}
template <typename T, int MODE, int LK, int SK> RadixFn<T> pass_row(int K)
{
    return pass_pick<T, MODE, false, LK, SK, 1, PASS_ROW_MAX>(K);
}
template <typename T, int MODE, int LK, int SK> RadixFn<T> pass_col(int K)
{
    return pass_pick<T, MODE, true, LK, SK, PASS_COL_MIN, PASS_COL_MAX>(K);
}

}  // namespace gfa
