"""The radix pass kernels at their edges: every number of row bits and column
bits, last tiles that are partly empty, tables of the other direction, and the
CKKS loads and stores.  Against the oracle, tolerances as in helpers.TOL."""
import numpy as np
import pytest

import oracle as O
from helpers import TOL, rel_err, rng_complex, to_dev, to_host

pytestmark = pytest.mark.gpu


def _g():
    import gpufft_amd as G
    return G


def _batch(n_power):
    # a full row tile of 2^12 elements and one transform more
    return (1 << (12 - n_power)) + 1 if n_power < 11 else 3 if n_power < 18 else 1


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n_power", list(range(1, 24)))
def test_c2c_every_size(prec, n_power):
    G = _g()
    batch, L = _batch(n_power), 1 << n_power
    rng = np.random.default_rng(50 + n_power)
    t = O.fft_tables(max(1, L // 2), prec)
    x = rng_complex(rng, batch * L, prec)
    d = to_dev(x)
    G.GPU_FFT(d, to_dev(t["rev"]), G.config(n_power, G.FORWARD), batch)
    ref = O.c2c_forward(x, n_power, batch, t["rev"], 0, prec)
    assert rel_err(to_host(d), ref) < TOL[prec]
    d = to_dev(ref)
    G.GPU_FFT(d, to_dev(t["inv_rev"]), G.config(n_power, G.INVERSE, mod_inverse=1.0 / L), batch)
    assert rel_err(to_host(d), x) < 4 * TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nega", [0, 1])
@pytest.mark.parametrize("n_power", [2, 4, 9, 13, 15, 18])
def test_c2c_other_direction_table(prec, nega, n_power):
    """FORWARD with the inverse table and INVERSE with the forward one: the
    transforms of the opposite exponent."""
    G = _g()
    batch, L = 2, 1 << n_power
    rng = np.random.default_rng(80 + n_power)
    t = O.fft_tables(L if nega else L // 2, prec)
    rp = G.X_N_PLUS if nega else G.X_N_MINUS
    x = rng_complex(rng, batch * L, prec)
    d = to_dev(x)
    G.GPU_FFT(d, to_dev(t["inv_rev"]), G.config(n_power, G.FORWARD, rp), batch)
    ref = O.c2c_forward(x, n_power, batch, t["inv_rev"], nega, prec)
    assert rel_err(to_host(d), ref) < TOL[prec]
    d = to_dev(x)
    G.GPU_FFT(d, to_dev(t["rev"]), G.config(n_power, G.INVERSE, rp), batch)
    ref = O.c2c_inverse(x, n_power, batch, t["rev"], nega, 0, complex(1.0), prec)
    assert rel_err(to_host(d), ref) < TOL[prec]


@pytest.mark.parametrize("inverse_table", [False, True])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n_power", [3, 4, 6, 7, 8, 9, 10, 16, 18, 19, 20])
def test_special_sizes_and_tables(prec, n_power, inverse_table):
    G = _g()
    batch, l = _batch(n_power), 1 << n_power
    rng = np.random.default_rng(110 + n_power)
    T = O.special_table(l, inverse_table, prec)
    z = rng_complex(rng, batch * l, prec)
    tol = TOL[prec] * (4 if prec == "f32" else 1)
    d = to_dev(z)
    G.GPU_Special_FFT(d, to_dev(T), G.config(n_power, G.FORWARD), batch)
    assert rel_err(to_host(d), O.special_forward(z, n_power, batch, T, prec)) < tol
    d = to_dev(z)
    G.GPU_Special_FFT(d, to_dev(T), G.config(n_power, G.INVERSE), batch)
    assert rel_err(to_host(d), O.special_inverse(z, n_power, batch, T, complex(1.0), prec)) < tol


@pytest.mark.parametrize("delta", [2.0 ** 30, 3.0 ** 17])
@pytest.mark.parametrize("n_power", [1, 2, 5, 10, 12, 13, 14, 16, 17, 18, 19, 20])
def test_ckks_sizes(n_power, delta):
    """Decode against the oracle, a power-of-two scale and another; the slots
    of integer coefficients encode to those integers."""
    import torch
    G = _g()
    batch, l = _batch(n_power), 1 << n_power
    rng = np.random.default_rng(140 + n_power)
    m = rng.integers(-(1 << 26), 1 << 26, size=batch * 2 * l)
    T, Ti = O.special_table(l), O.special_table(l, True)
    slots = torch.empty(batch * l, dtype=torch.complex128, device="cuda")
    G.ckks_decode(to_dev(m), slots, to_dev(T), n_power, delta, batch)
    assert rel_err(to_host(slots), O.ckks_decode(m, n_power, batch, T, delta)) < TOL["f64"]
    coeffs = torch.empty(batch * 2 * l, dtype=torch.int64, device="cuda")
    work = torch.empty(batch * l, dtype=torch.complex128, device="cuda")
    G.ckks_encode(slots, coeffs, to_dev(Ti), n_power, delta, batch, work)
    assert np.array_equal(to_host(coeffs), m)
