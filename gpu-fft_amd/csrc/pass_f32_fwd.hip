// Standard forward passes, float.
#include "passes.hpp"

namespace gfa {

template <> RadixFn<float> pass_std_fwd<float>(bool col, int K, int lk, int sk)
{
    if (sk != ST_CPLX) return nullptr;
#define GFA_SEL(L) \
    if (lk == L) return col ? pass_col<float, MODE_STD_FWD, L, ST_CPLX>(K) : pass_row<float, MODE_STD_FWD, L, ST_CPLX>(K);
    GFA_SEL(LD_CPLX)
    GFA_SEL(LD_REAL)
    GFA_SEL(LD_FOLD)
#undef GFA_SEL
    return nullptr;
}

}  // namespace gfa
