"""Special tables of another primitive root (every entry raised to an odd power):
the transforms are the networks of the table that is passed, so the results
are the oracle's for that table.  Tolerances as in helpers.TOL."""
import numpy as np
import pytest

import oracle as O
from helpers import TOL, cdtype, rel_err, rng_complex, to_dev, to_host

pytestmark = pytest.mark.gpu


def _g():
    import gpufft_amd as G
    return G


@pytest.mark.parametrize("power", [3, 5, 7])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n_power", [1, 2, 4, 7, 8, 10, 13, 14, 17, 20])
def test_special(n_power, prec, power):
    G = _g()
    batch, l = 2, 1 << n_power
    rng = np.random.default_rng(8700 + n_power)
    T = (O.special_table(l) ** power).astype(cdtype(prec))
    z = rng_complex(rng, batch * l, prec)
    tol = TOL[prec] * (4 if prec == "f32" else 1)
    d = to_dev(z)
    G.GPU_Special_FFT(d, to_dev(T), G.config(n_power, G.FORWARD), batch)
    assert rel_err(to_host(d), O.special_forward(z, n_power, batch, T, prec)) < tol
    d = to_dev(z)
    G.GPU_Special_FFT(d, to_dev(T), G.config(n_power, G.INVERSE), batch)
    assert rel_err(to_host(d), O.special_inverse(z, n_power, batch, T, complex(1.0), prec)) < tol


@pytest.mark.parametrize("power", [3, 5])
@pytest.mark.parametrize("n_power", [3, 14, 18])
def test_ckks_decode(n_power, power):
    import torch
    G = _g()
    batch, l = 2, 1 << n_power
    rng = np.random.default_rng(8800 + n_power)
    m = rng.integers(-(1 << 26), 1 << 26, size=batch * 2 * l)
    T = O.special_table(l) ** power
    slots = torch.empty(batch * l, dtype=torch.complex128, device="cuda")
    G.ckks_decode(to_dev(m), slots, to_dev(T), n_power, 2.0 ** 30, batch)
    assert rel_err(to_host(slots), O.ckks_decode(m, n_power, batch, T, 2.0 ** 30)) < TOL["f64"]
