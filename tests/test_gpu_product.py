"""The fused FP64 product kernels: every ring size, with one product, with a
last workgroup that is partly empty, and with more products than the
persistent workgroups take in one round.  Rounded products against the exact
ones of the oracle's NTT."""
import numpy as np
import pytest

import oracle as O
from helpers import SEED_BASE, to_dev, to_host

pytestmark = pytest.mark.gpu

# products that 256 CUs take at once, by ring power
ROUND = {7: 32768, 8: 16384, 9: 8192, 10: 4096, 11: 2048, 12: 1024, 13: 512, 14: 256, 15: 128, 16: 64,
         17: 32}


@pytest.mark.parametrize("which", ["one", "ragged", "rounds"])
@pytest.mark.parametrize("ring_power", sorted(ROUND))
def test_product_exact(ring_power, which):
    import torch

    import gpufft_amd as G
    N = 1 << ring_power
    batch = {"one": 1, "ragged": 67, "rounds": 2 * ROUND[ring_power] + 5}[which]
    if which == "ragged" and ring_power > 13:
        batch = 9  # a second group of eight, partly empty
    a = O.fill_uniform(SEED_BASE + 7 * ring_power, 0, 1 << 20, batch * N)
    b = O.fill_uniform(SEED_BASE + 7 * ring_power + 1, -128, 129, batch * N)
    plan = G.PolymulPlan(ring_power, G.PREC_F64, max_batch=batch)
    out = torch.full((batch * N + 8,), -0.25, dtype=torch.float64, device="cuda")
    plan.multiply_f64(to_dev(a.astype(np.float64)), to_dev(b.astype(np.float64)), out, batch)
    got = to_host(out)
    plan.close()
    exact = O.ntt_negacyclic(a.reshape(batch, N), b.reshape(batch, N)).reshape(-1)
    assert np.array_equal(np.round(got[:batch * N]).astype(np.int64), exact)
    assert np.max(np.abs(got[:batch * N] - exact)) < 1e-3
    assert np.all(got[batch * N:] == -0.25)  # nothing beyond the batch


@pytest.mark.parametrize("ring_power", [9, 13, 14, 16])
def test_product_in_place_and_captured(ring_power):
    """out may be one of the operands; a captured call replays to the same
    bits as the eager one."""
    import torch

    import gpufft_amd as G
    N, batch = 1 << ring_power, 5
    a = to_dev(O.fill_uniform(SEED_BASE + 51, 0, 1 << 20, batch * N).astype(np.float64))
    b = to_dev(O.fill_uniform(SEED_BASE + 52, -128, 129, batch * N).astype(np.float64))
    plan = G.PolymulPlan(ring_power, G.PREC_F64, max_batch=batch)
    ref = torch.empty_like(a)
    plan.multiply_f64(a, b, ref, batch)
    inplace = a.clone()
    plan.multiply_f64(inplace, b, inplace, batch)
    assert torch.equal(inplace, ref)
    out = torch.empty_like(a)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        plan.multiply_f64(a, b, out, batch, stream=s.cuda_stream)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        plan.multiply_f64(a, b, inplace, batch)  # eager work in between
    plan.close()
