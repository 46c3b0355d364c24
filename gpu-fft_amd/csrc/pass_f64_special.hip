// Special passes, double, with the CKKS loads and stores.
#include "passes.hpp"

namespace gfa {

template <> RadixFn<double> pass_spe_fwd<double>(bool col, int K, int lk, int sk)
{
    if (sk != ST_CPLX) return nullptr;
    if (lk == LD_CPLX)
        return col ? pass_col<double, MODE_SPE_FWD, LD_CPLX, ST_CPLX>(K)
                   : pass_row<double, MODE_SPE_FWD, LD_CPLX, ST_CPLX>(K);
    if (lk == LD_CKKS && !col) return pass_row<double, MODE_SPE_FWD, LD_CKKS, ST_CPLX>(K);
    return nullptr;
}

template <> RadixFn<double> pass_spe_inv<double>(bool col, int K, int lk, int sk)
{
    if (lk != LD_CPLX) return nullptr;
    if (sk == ST_CPLX)
        return col ? pass_col<double, MODE_SPE_INV, LD_CPLX, ST_CPLX>(K)
                   : pass_row<double, MODE_SPE_INV, LD_CPLX, ST_CPLX>(K);
    if (sk == ST_CKKS && !col) return pass_row<double, MODE_SPE_INV, LD_CPLX, ST_CKKS>(K);
    return nullptr;
}

}  // namespace gfa
