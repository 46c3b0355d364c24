// Standard inverse passes, double.
#include "passes.hpp"

namespace gfa {

template <> RadixFn<double> pass_std_inv<double>(bool col, int K, int lk, int sk)
{
#define GFA_ROW(L, S) \
    if (!col && lk == L && sk == S) return pass_row<double, MODE_STD_INV, L, S>(K);
    GFA_ROW(LD_CPLX, ST_CPLX)
    GFA_ROW(LD_CPLX, ST_REAL)
    GFA_ROW(LD_CPLX, ST_UNFOLD)
    GFA_ROW(LD_MUL, ST_CPLX)
    GFA_ROW(LD_MUL, ST_REAL)
    GFA_ROW(LD_MUL, ST_UNFOLD)
    GFA_ROW(LD_RR_PACK, ST_CPLX)
#undef GFA_ROW
#define GFA_COL(S) \
    if (col && lk == LD_CPLX && sk == S) return pass_col<double, MODE_STD_INV, LD_CPLX, S>(K);
    GFA_COL(ST_CPLX)
    GFA_COL(ST_REAL)
    GFA_COL(ST_UNFOLD)
#undef GFA_COL
    return nullptr;
}

}  // namespace gfa
