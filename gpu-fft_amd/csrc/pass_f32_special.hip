// Special passes, float, with the hi/lo split loads and the double sum store.
#include "passes.hpp"

namespace gfa {

template <> RadixFn<float> pass_spe_fwd<float>(bool col, int K, int lk, int sk)
{
#define GFA_ROW(L, S) \
    if (!col && lk == L && sk == S) return pass_row<float, MODE_SPE_FWD, L, S>(K);
    GFA_ROW(LD_CPLX, ST_CPLX)
    GFA_ROW(LD_SPLIT_HI, ST_CPLX)
    GFA_ROW(LD_SPLIT_LO, ST_CPLX)
    GFA_ROW(LD_SPLIT_LO, ST_SUM_F64)
#undef GFA_ROW
    if (col && lk == LD_CPLX && sk == ST_CPLX) return pass_col<float, MODE_SPE_FWD, LD_CPLX, ST_CPLX>(K);
    if (col && lk == LD_CPLX && sk == ST_SUM_F64)
        return pass_col<float, MODE_SPE_FWD, LD_CPLX, ST_SUM_F64>(K);
    return nullptr;
}

template <> RadixFn<float> pass_spe_inv<float>(bool col, int K, int lk, int sk)
{
#define GFA_ROW(L, S) \
    if (!col && lk == L && sk == S) return pass_row<float, MODE_SPE_INV, L, S>(K);
    GFA_ROW(LD_CPLX, ST_CPLX)
    GFA_ROW(LD_CPLX, ST_SUM_F64)
    GFA_ROW(LD_SPLIT_HI, ST_CPLX)
    GFA_ROW(LD_SPLIT_LO, ST_SUM_F64)
#undef GFA_ROW
#define GFA_COL(L) \
    if (col && lk == L && sk == ST_CPLX) return pass_col<float, MODE_SPE_INV, L, ST_CPLX>(K);
    GFA_COL(LD_CPLX)
    GFA_COL(LD_SPLIT_HI)
    GFA_COL(LD_SPLIT_LO)
#undef GFA_COL
    return nullptr;
}

}  // namespace gfa
