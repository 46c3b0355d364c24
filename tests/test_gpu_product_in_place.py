"""Fused FP64 products whose output is one of the operands, with more products
than the persistent workgroups take at once: a workgroup loads operands of its
next product before it stores the current one.  The bits of a call with an
output of its own."""
import numpy as np
import pytest

import oracle as O
from helpers import SEED_BASE, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("operand", ["a", "b"])
@pytest.mark.parametrize("ring_power,batch", [(9, 16387), (11, 2051), (13, 1030), (14, 517), (16, 131)])
def test_out_is_operand(ring_power, batch, operand):
    import torch

    import gpufft_amd as G
    N = 1 << ring_power
    a = to_dev(O.fill_uniform(SEED_BASE + 61, 0, 1 << 20, batch * N).astype(np.float64))
    b = to_dev(O.fill_uniform(SEED_BASE + 62, -128, 129, batch * N).astype(np.float64))
    plan = G.PolymulPlan(ring_power, G.PREC_F64, max_batch=batch)
    ref = torch.empty_like(a)
    plan.multiply_f64(a, b, ref, batch)
    out = (a if operand == "a" else b).clone()
    if operand == "a":
        plan.multiply_f64(out, b, out, batch)
    else:
        plan.multiply_f64(a, out, out, batch)
    assert torch.equal(out, ref)
    plan.close()
