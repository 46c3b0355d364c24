"""R_R and FFNT calls with tables of the other direction: FORWARD with the
inverse tables and INVERSE with the forward ones are the transforms of the
opposite exponent, at every size and batch, whichever kernels a call takes; and
with the table of another root.
Against the oracle, tolerances as in helpers.TOL."""
import numpy as np
import pytest

import oracle as O
from helpers import TOL, cdtype, rdtype, rel_err, rng_complex, to_dev, to_host

pytestmark = pytest.mark.gpu

# batches on both sides of the lines between the kernels, 256 compute units
FORWARD = [("f64", 13, 3), ("f64", 14, 1), ("f64", 14, 128), ("f64", 14, 130), ("f64", 14, 184),
           ("f64", 14, 185), ("f64", 15, 2), ("f64", 15, 3), ("f64", 15, 64), ("f64", 15, 65),
           ("f64", 15, 88), ("f64", 15, 89), ("f64", 16, 2), ("f64", 16, 3), ("f64", 16, 48), ("f64", 16, 49),
           ("f64", 16, 8), ("f64", 16, 9), ("f64", 16, 32), ("f64", 16, 33), ("f64", 16, 64),
           ("f64", 16, 65), ("f64", 17, 2),
           ("f32", 14, 3), ("f32", 15, 16), ("f32", 15, 17), ("f32", 15, 33), ("f32", 16, 16),
           ("f32", 16, 17), ("f32", 16, 64), ("f32", 16, 65), ("f32", 16, 81), ("f32", 17, 8), ("f32", 17, 9),
           ("f32", 17, 33), ("f32", 17, 41)]


def _g():
    import gpufft_amd as G
    return G


def _tables(kind, nega, L, prec):
    """(twist, root) of the forward and of the inverse."""
    if kind == "r2r":
        t = O.fft_tables(L if nega else L // 2, prec)
        return (None, t["rev"]), (None, t["inv_rev"])
    t = O.ffnt_tables(2 * L, prec)
    return (t["twist"], t["rev_root"]), (t["untwist"], t["inv_rev_root"])


@pytest.mark.parametrize("kind,nega,which", [("r2r", 0, "root"), ("r2r", 1, "root"), ("ffnt", 0, "both"),
                                             ("ffnt", 0, "root"), ("r2r", 0, "none"), ("r2r", 1, "none"),
                                             ("ffnt", 0, "none")])
@pytest.mark.parametrize("prec,n,batch", FORWARD)
def test_forward_with_inverse_tables(prec, n, batch, kind, nega, which):
    """which: both tables of the other direction, the root table alone, or
    none (the forward's own, on both sides of the same lines)."""
    import torch
    G = _g()
    L = 1 << n
    R = L if kind == "r2r" else 2 * L
    rng = np.random.default_rng(8000 + 16 * n + batch)
    real = rng.standard_normal(batch * R).astype(rdtype(prec))
    rows = sorted({0, batch // 2, batch - 1})
    some = np.concatenate([real[k * R:(k + 1) * R] for k in rows])
    fwd, inv = _tables(kind, nega, L, prec)
    twist, root = (inv if which == "both" else fwd)[0], (fwd if which == "none" else inv)[1]
    dt = torch.empty(batch * L, dtype=torch.complex128 if prec == "f64" else torch.complex64, device="cuda")
    if kind == "r2r":
        rp = G.X_N_PLUS if nega else G.X_N_MINUS
        G.GPU_FFT_R(to_dev(real), dt, to_dev(root), G.config(n, G.FORWARD, rp), batch)
        ref = O.r2r_forward(some, n, len(rows), root, nega, prec)
    else:
        G.GPU_FFNT(to_dev(real), dt, to_dev(twist), to_dev(root), G.config(n + 1, G.FORWARD), batch)
        ref = O.ffnt_forward(some, n + 1, len(rows), twist, root, prec)
    got = to_host(dt)
    got = np.concatenate([got[k * L:(k + 1) * L] for k in rows])
    assert rel_err(got, ref) < TOL[prec]


@pytest.mark.parametrize("mult", [0, 1])
@pytest.mark.parametrize("kind,nega", [("r2r", 0), ("r2r", 1), ("ffnt", 0)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [13, 14, 15, 16, 17])
def test_inverse_with_forward_tables(n, prec, kind, nega, mult):
    import torch
    G = _g()
    batch, L = 3, 1 << n
    R = L if kind == "r2r" else 2 * L
    rng = np.random.default_rng(8500 + n)
    temp = rng_complex(rng, 2 * batch * L, prec)
    (twist, root), _ = _tables(kind, nega, L, prec)
    out = torch.empty(batch * R, dtype=torch.float64 if prec == "f64" else torch.float32, device="cuda")
    if kind == "r2r":
        rp = G.X_N_PLUS if nega else G.X_N_MINUS
        G.GPU_FFT_R(out, to_dev(temp), to_dev(root), G.config(n, G.INVERSE, rp, 1.0 / L), batch, bool(mult))
        ref = O.r2r_inverse(temp, n, batch, root, nega, mult, complex(1.0 / L), prec)
    else:
        G.GPU_FFNT(out, to_dev(temp), to_dev(twist), to_dev(root),
                   G.config(n + 1, G.INVERSE, mod_inverse=1.0 / L), batch, bool(mult))
        ref = O.ffnt_inverse(temp, n + 1, batch, twist, root, mult, complex(1.0 / L), prec)
    assert rel_err(to_host(out), ref) < TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nega", [0, 1])
@pytest.mark.parametrize("n_power,batch", [(4, 2), (13, 2), (18, 2), (14, 130), (16, 33)])
def test_other_root(n_power, batch, nega, prec):
    """C_C and R_R FORWARD with a table of another primitive root (the third
    powers), the last transform of the batch."""
    import torch
    G = _g()
    L = 1 << n_power
    rng = np.random.default_rng(8900 + n_power)
    T = (O.fft_tables(L if nega else L // 2, "f64")["rev"] ** 3).astype(cdtype(prec))
    rp = G.X_N_PLUS if nega else G.X_N_MINUS
    x = rng_complex(rng, batch * L, prec)
    d = to_dev(x)
    G.GPU_FFT(d, to_dev(T), G.config(n_power, G.FORWARD, rp), batch)
    ref = O.c2c_forward(x[-L:], n_power, 1, T, nega, prec)
    assert rel_err(to_host(d)[-L:], ref) < TOL[prec]
    real = np.ascontiguousarray(x.real)
    d = torch.empty(batch * L, dtype=torch.complex128 if prec == "f64" else torch.complex64, device="cuda")
    G.GPU_FFT_R(to_dev(real), d, to_dev(T), G.config(n_power, G.FORWARD, rp), batch)
    ref = O.r2r_forward(real[-L:], n_power, 1, T, nega, prec)
    assert rel_err(to_host(d)[-L:], ref) < TOL[prec]
