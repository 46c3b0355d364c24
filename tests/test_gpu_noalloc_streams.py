"""Overlapping calls of gpufft_polymul_f64_noalloc on two streams: rings up to 2^14
share the library's root table, whose values must not depend on the ring, so
every call gives the bits of a call alone."""
import ctypes

import numpy as np
import pytest

import oracle as O
from helpers import SEED_BASE, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rings", [(7, 14), (10, 13), (12, 14), (14, 16)])
def test_overlapping_rings(rings):
    import torch

    import gpufft_amd as G
    f = G.lib().gpufft_polymul_f64_noalloc
    f.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int, ctypes.c_int] + [ctypes.c_void_p] * 5
    f.restype = ctypes.c_int
    calls, batch = 60, 2

    def setup(ring, seed):
        N = 1 << ring
        a = to_dev(O.fill_uniform(SEED_BASE + seed, 0, 1 << 20, batch * N).astype(np.float64))
        b = to_dev(O.fill_uniform(SEED_BASE + seed + 1, -128, 129, batch * N).astype(np.float64))
        tabs = [G.generate_table(k, ring - 1, inv) for k in (G.TABLE_FFNT_TWIST, G.TABLE_FFNT_ROOT)
                for inv in (False, True)]
        outs = [torch.full_like(a, -1.0) for _ in range(calls + 1)]
        ptrs = [t.data_ptr() for t in tabs]

        def run(k, stream):
            G.check(f(a.data_ptr(), b.data_ptr(), outs[k].data_ptr(), ring, batch, *ptrs, stream))
        return run, outs, tabs

    sides = [setup(r, 700 + 10 * i) for i, r in enumerate(rings)]
    streams = [torch.cuda.Stream() for _ in rings]
    torch.cuda.synchronize()
    for run, _, _ in sides:  # alone
        run(calls, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    for k in range(calls):
        for (run, _, _), s in zip(sides, streams):
            run(k, s.cuda_stream)
    torch.cuda.synchronize()
    for ring, (_, outs, _) in zip(rings, sides):
        want = to_host(outs[calls])
        for k in range(calls):
            assert np.array_equal(to_host(outs[k]), want), (ring, k)
