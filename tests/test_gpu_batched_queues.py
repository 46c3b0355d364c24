"""The work queues of the batched kernel: lists shorter than the queues and the
grid, and grids of one workgroup up to more than the items, launched several
times in a row (the last workgroup clears the counters for the next launch).
Every launch gives the exact products of the oracle's NTT."""
import numpy as np
import pytest

import oracle as O
from helpers import SEED_BASE, to_dev, to_host

pytestmark = pytest.mark.gpu

RING = 8


@pytest.mark.parametrize("prec", ["f64", "split"])
@pytest.mark.parametrize("grid", [1, 7, 8, 9, 256])
@pytest.mark.parametrize("count", [1, 7, 8, 9, 70])
def test_short_lists(count, grid, prec):
    import torch

    import gpufft_amd as G
    N = 1 << RING
    descs, n_in, n_out = G.pack_products([G.PRODUCT_NEGACYCLIC] * count, [RING] * count)
    assert n_in == n_out == count * N
    a = O.fill_uniform(SEED_BASE + 801, -256, 256, n_in)
    b = O.fill_uniform(SEED_BASE + 802, -256, 256, n_in)
    exact = O.ntt_negacyclic(a.reshape(count, N), b.reshape(count, N)).reshape(-1)
    plan = G.BatchedPlan(descs, precision=G.PREC_F64) if prec == "f64" else G.BatchedPlan(descs, 5, 2, 5, 2)
    plan.set_tuning(4, grid)
    da, db = to_dev(a.astype(np.int32)), to_dev(b.astype(np.int32))
    outs = [torch.full((n_out,), -7, dtype=torch.int64, device="cuda") for _ in range(4)]
    torch.cuda.synchronize()
    for out in outs:
        plan.execute(da, db, out)
    got = [to_host(o) for o in outs]
    plan.close()
    for g in got:
        assert np.array_equal(g, exact)
