"""The one-launch R_R and FFNT forward of double transforms at the edges of its
dispatch: the last batch that goes to one workgroup per sub-problem, the first
that goes to the persistent workgroups, one that takes them several rounds with
a partial last group, and an input that is aligned to 8 bytes only.  Against
the oracle, tolerance as in helpers.TOL."""
import numpy as np
import pytest

import oracle as O
from helpers import TOL, rel_err, to_dev, to_host

pytestmark = pytest.mark.gpu

# transforms of 2^n points that 256 workgroups take at once
ROUND = {14: 128, 15: 64, 16: 32}


@pytest.mark.parametrize("which", ["last", "first", "rounds"])
@pytest.mark.parametrize("kind,nega", [("r2r", 0), ("r2r", 1), ("ffnt", 1)])
@pytest.mark.parametrize("n", [14, 15, 16])
def test_forward_large_batches(n, kind, nega, which):
    import torch

    import gpufft_amd as G
    batch = {"last": ROUND[n], "first": ROUND[n] + 2, "rounds": 2 * ROUND[n] + 10}[which]
    L = 1 << n
    real_len = L if kind == "r2r" else 2 * L
    rng = np.random.default_rng(7000 + n * 4 + nega * 2 + (kind == "ffnt"))
    real = rng.standard_normal(batch * real_len)
    room = torch.zeros(batch * real_len + 1, dtype=torch.float64, device="cuda")
    dr = room[1:]
    dr.copy_(to_dev(real))
    dt = torch.full((batch * L + 8,), -0.25, dtype=torch.complex128, device="cuda")
    if kind == "r2r":
        tab = O.fft_tables(L if nega else L // 2, "f64")["rev"]
        G.GPU_FFT_R(dr, dt, to_dev(tab), G.config(n, G.FORWARD, G.X_N_PLUS if nega else G.X_N_MINUS), batch)
        ref = O.r2r_forward(real, n, batch, tab, nega, "f64")
    else:
        t = O.ffnt_tables(2 * L, "f64")
        G.GPU_FFNT(dr, dt, to_dev(t["twist"]), to_dev(t["rev_root"]), G.config(n + 1, G.FORWARD), batch)
        ref = O.ffnt_forward(real, n + 1, batch, t["twist"], t["rev_root"], "f64")
    got = to_host(dt)
    assert rel_err(got[:batch * L], ref) < TOL["f64"]
    assert np.all(got[batch * L:] == -0.25)  # nothing beyond the batch


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["r2r", "ffnt"])
@pytest.mark.parametrize("n", [14, 15, 16, 17])
def test_batches_agree(prec, kind, n):
    """A batch and its transforms one call each may run different kernels: the
    same results within rounding, both directions."""
    import torch

    import gpufft_amd as G
    batch, L = 34, 1 << n
    real_len = L if kind == "r2r" else 2 * L
    rdt = torch.float64 if prec == "f64" else torch.float32
    cdt = torch.complex128 if prec == "f64" else torch.complex64
    rng = np.random.default_rng(7100 + n)
    dr = to_dev(rng.standard_normal(batch * real_len).astype(np.float64 if prec == "f64" else np.float32))
    cfg_n = n if kind == "r2r" else n + 1
    if kind == "r2r":
        t = O.fft_tables(L // 2, prec)
        f, i = to_dev(t["rev"]), to_dev(t["inv_rev"])
    else:
        t = O.ffnt_tables(2 * L, prec)
        f, i, tw, un = (to_dev(t[k]) for k in ("rev_root", "inv_rev_root", "twist", "untwist"))

    def run(r, d, cfg, b):
        if kind == "r2r":
            G.GPU_FFT_R(r, d, f if cfg is fwd else i, cfg, b)
        else:
            G.GPU_FFNT(r, d, tw if cfg is fwd else un, f if cfg is fwd else i, cfg, b)

    fwd, inv = G.config(cfg_n, G.FORWARD), G.config(cfg_n, G.INVERSE, mod_inverse=1.0 / L)
    many, one = (torch.empty(batch * L, dtype=cdt, device="cuda") for _ in range(2))
    run(dr, many, fwd, batch)
    for k in (0, 17, batch - 1):
        run(dr[k * real_len:], one[k * L:], fwd, 1)
        a, b = to_host(many[k * L:(k + 1) * L]), to_host(one[k * L:(k + 1) * L])
        assert rel_err(a, b) < 2 * TOL[prec]
    src, back, back1 = many.clone(), torch.empty_like(dr), torch.empty_like(dr)
    run(back, src, inv, batch)
    for k in (0, 17, batch - 1):
        run(back1[k * real_len:], many[k * L:(k + 1) * L].clone(), inv, 1)
        s = slice(k * real_len, (k + 1) * real_len)
        assert rel_err(to_host(back[s]), to_host(back1[s])) < 8 * TOL[prec]
        assert rel_err(to_host(back[s]), to_host(dr[s])) < 8 * TOL[prec]
