"""The calls that programs built on this framework spend their GPU time in.

Each case is one of the public operations at one size.  Integer polynomials go
in as a caller holds them (doubles, floats or int32), products come out whole.

  polymul_f64     fused FP64 products mod X^N + 1 through a plan
  polymul_split   exact int32 -> int64 products mod X^N + 1 (FP32 limbs)
  ffnt_product    GPU_FFNT forward on both operands, inverse with the product
  rr_product      GPU_FFT on real data, forward on both, inverse with the product
  c2c_product     GPU_FFT in place on complex data, same flow, X^N -+ 1
  c2c_round       GPU_FFT in place, forward then inverse (spectral filtering)
  special_round   GPU_Special_FFT in place, inverse (encode side) then forward
  ckks            CKKS decode of integer coefficients and encode of the slots
  batched         a list of products of uneven ring sizes, one plan
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gpu-fft_amd"))

import gpufft_amd as G  # noqa: E402


def listed():
    return [
        # one product of degree < 2^12 operands, padded to the ring 2^13: the
        # interactive call, all latency
        {"name": "polymul_f64_one", "op": "polymul_f64", "ring": 13, "batch": 1},
        # a ragged batch at a lattice-cryptography ring that fits one workgroup
        {"name": "polymul_f64_ring14", "op": "polymul_f64", "ring": 14, "batch": 331},
        # the headline workload: N = 2^16, batch 256
        {"name": "polymul_f64_ring16", "op": "polymul_f64", "ring": 16, "batch": 256},
        # the headline workload with exact integer outputs from FP32 limbs
        {"name": "polymul_split_ring16", "op": "polymul_split", "ring": 16, "batch": 256},
        # the two-call drop-in flow at the headline size
        {"name": "ffnt_f64_ring16", "op": "ffnt_product", "prec": "f64", "ring": 16, "batch": 256},
        # bootstrapping-sized float products in a large odd batch
        {"name": "ffnt_f32_ring11", "op": "ffnt_product", "prec": "f32", "ring": 11, "batch": 1501},
        # cyclic products of zero-padded real operands, N = 2^16, batch 64
        {"name": "rr_f64_n16", "op": "rr_product", "prec": "f64", "n": 16, "batch": 64},
        # one complex cyclic product of 4096-coefficient operands
        {"name": "c2c_f64_n13", "op": "c2c_product", "prec": "f64", "n": 13, "batch": 1, "nega": 0},
        # a few long float transforms there and back
        {"name": "c2c_f32_n20", "op": "c2c_round", "prec": "f32", "n": 20, "batch": 5},
        # one very long double transform there and back
        {"name": "c2c_f64_n23", "op": "c2c_round", "prec": "f64", "n": 23, "batch": 1},
        # CKKS decode and encode of 512 ciphertexts' worth of 2^15 slots
        {"name": "ckks_n15", "op": "ckks", "n": 15, "batch": 512},
        # 1000 FP64 products of rings 2^10 .. 2^17, half linear, half negacyclic
        {"name": "batched_f64_1000", "op": "batched", "prec": "f64", "count": 1000},
    ]


# log2 of the sizes a drawn case takes and of the elements (size x batch) it
# may reach; every size in the range is used, the batch is what varies most
RANGES = {
    "polymul_f64": (7, 17, 24),
    "polymul_split": (8, 17, 23),
    "ffnt_product": (6, 21, 24),
    "rr_product": (5, 21, 22),
    "c2c_product": (5, 21, 22),
    "c2c_round": (10, 23, 23),
    "special_round": (8, 17, 23),
    "ckks": (8, 17, 23),
}
MAX_BATCH = 4096


def draw(rng):
    op = rng.choice(sorted(RANGES) + ["batched", "polymul_f64", "ffnt_product", "c2c_product"])
    if op == "batched":
        return {"op": op, "prec": rng.choice(["f64", "split"]),
                "count": int(round(math.exp(rng.uniform(math.log(3), math.log(700)))))}
    lo, hi, total = RANGES[op]
    n = rng.randint(lo, hi)
    most = min(MAX_BATCH, 1 << (total - n)) if total > n else 1
    batch = max(1, min(most, int(round(math.exp(rng.uniform(0.0, math.log(most)))))))
    case = {"op": op, "batch": batch}
    case["ring" if op in ("polymul_f64", "polymul_split", "ffnt_product") else "n"] = n
    if op in ("ffnt_product", "rr_product", "c2c_product", "c2c_round", "special_round"):
        case["prec"] = rng.choice(["f64", "f32"])
    if op == "c2c_product":
        case["nega"] = rng.choice([0, 1])
    return case


# ---- inputs ----
def _ints(gen, lo, hi, count, dtype):
    """Integers uniform in [lo, hi), as dtype, on the GPU."""
    v = torch.randint(lo, hi, (count,), generator=gen, device="cuda", dtype=torch.int32)
    return v if dtype == torch.int32 else v.to(dtype)


def _bounds(case):
    """Coefficient ranges of the two operands: the headline's for double and
    integer products, small digits for float ones."""
    if case.get("prec") == "f32":
        return (-8, 8), (-8, 8)
    if case["op"] in ("rr_product", "c2c_product"):
        return (-1024, 1024), (-1024, 1024)
    if case["op"] == "batched":
        return (-256, 256), (-256, 256)
    return (0, 1 << 20), (-128, 129)


def _types(case):
    f32 = case.get("prec") == "f32"
    return (torch.float32, torch.complex64) if f32 else (torch.float64, torch.complex128)


def _operands(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    (alo, ahi), (blo, bhi) = _bounds(case)
    op = case["op"]
    if op == "batched":
        kinds, rings = _list(case)
        count = sum(1 << r for r in rings)
        return (_ints(gen, alo, ahi, count, torch.int32), _ints(gen, blo, bhi, count, torch.int32))
    size = case["ring"] if "ring" in case else case["n"]
    count = case["batch"] << size
    dtype = torch.int32 if op == "polymul_split" else _types(case)[0]
    a, b = _ints(gen, alo, ahi, count, dtype), _ints(gen, blo, bhi, count, dtype)
    if op in ("rr_product", "c2c_product") and not case.get("nega"):
        # cyclic products of zero-padded operands
        for v in (a, b):
            v.view(case["batch"], -1)[:, 1 << (size - 1):] = 0
    return a, b


def _signal(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rdt, cdt = _types(case)
    return torch.randn(case["batch"] << case["n"], generator=gen, device="cuda", dtype=cdt)


def _coeffs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-(1 << 26), 1 << 26, (case["batch"] << (case["n"] + 1),), generator=gen,
                         device="cuda", dtype=torch.int64)


def _list(case):
    """Kinds and ring sizes of a list, a property of the case: rings uniform
    in 2^10 .. 2^17, every other product linear."""
    r = random.Random(case["count"])
    rings = [r.randint(10, 17) for _ in range(case["count"])]
    kinds = [G.PRODUCT_LINEAR if i % 2 == 0 else G.PRODUCT_NEGACYCLIC for i in range(case["count"])]
    return kinds, rings


# ---- the calls ----
def prepare(case, seed):
    op = case["op"]
    s = {"op": op, "batch": case.get("batch")}
    B = case.get("batch")
    if op in ("polymul_f64", "polymul_split"):
        s["a"], s["b"] = _operands(case, seed)
        if op == "polymul_f64":
            s["plan"] = G.PolymulPlan(case["ring"], G.PREC_F64, B)
            s["out"] = torch.empty(B << case["ring"], dtype=torch.float64, device="cuda")
        else:
            # a in [0, 2^20) as a - 2^19 in 5 digits of 4 bits, b whole
            s["plan"] = G.PolymulPlan(case["ring"], G.PREC_F32_SPLIT, B, 4, 5, 0, 1)
            s["plan"].a_center_log2 = 19
            s["out"] = torch.empty(B << case["ring"], dtype=torch.int64, device="cuda")
    elif op == "ffnt_product":
        n, p = case["ring"], case["prec"]
        rdt, cdt = _types(case)
        s["real"] = torch.cat(_operands(case, seed))
        s["temp"] = torch.empty(B << n, dtype=cdt, device="cuda")
        s["out"] = torch.empty(B << n, dtype=rdt, device="cuda")
        s["tables"] = [G.generate_table(k, n - 1, inv, prec=p)
                       for inv in (False, True) for k in (G.TABLE_FFNT_TWIST, G.TABLE_FFNT_ROOT)]
        s["fwd"] = G.config(n, G.FORWARD)
        s["inv"] = G.config(n, G.INVERSE, mod_inverse=2.0 / (1 << n))
    elif op == "rr_product":
        n, p = case["n"], case["prec"]
        rdt, cdt = _types(case)
        s["real"] = torch.cat(_operands(case, seed))
        s["temp"] = torch.empty(2 * B << n, dtype=cdt, device="cuda")
        s["out"] = torch.empty(B << n, dtype=rdt, device="cuda")
        s["tables"] = [G.generate_table(G.TABLE_FFT, n - 1, inv, prec=p) for inv in (False, True)]
        s["fwd"] = G.config(n, G.FORWARD)
        s["inv"] = G.config(n, G.INVERSE, mod_inverse=1.0 / (1 << n))
    elif op in ("c2c_product", "c2c_round"):
        n, p = case["n"], case["prec"]
        nega = case.get("nega", 0)
        poly = G.X_N_PLUS if nega else G.X_N_MINUS
        s["tables"] = [G.generate_table(G.TABLE_FFT, n if nega else n - 1, inv, prec=p)
                       for inv in (False, True)]
        s["fwd"] = G.config(n, G.FORWARD, poly)
        s["inv"] = G.config(n, G.INVERSE, poly, 1.0 / (1 << n))
        if op == "c2c_product":
            s["src"] = torch.cat(_operands(case, seed)).to(_types(case)[1])
            s["x"] = torch.empty_like(s["src"])
            s["product"] = s["x"][:B << n]
        else:
            s["x"] = _signal(case, seed)
    elif op == "special_round":
        n, p = case["n"], case["prec"]
        s["x"] = _signal(case, seed)
        s["tables"] = [G.generate_table(G.TABLE_SPECIAL, n, inv, prec=p) for inv in (False, True)]
        s["fwd"] = G.config(n, G.FORWARD)
        s["inv"] = G.config(n, G.INVERSE, mod_inverse=1.0 / (1 << n))
    elif op == "ckks":
        n = case["n"]
        s["n"] = n
        s["m"] = _coeffs(case, seed)
        s["coeffs"] = torch.empty_like(s["m"])
        s["slots"] = torch.empty(B << n, dtype=torch.complex128, device="cuda")
        s["work"] = torch.empty_like(s["slots"])
        s["tables"] = [G.generate_table(G.TABLE_SPECIAL, n, inv) for inv in (False, True)]
    else:
        s["a"], s["b"] = _operands(case, seed)
        descs, _, n_out = G.pack_products(*_list(case))
        if case["prec"] == "f64":
            s["plan"] = G.BatchedPlan(descs, precision=G.PREC_F64)
        else:
            s["plan"] = G.BatchedPlan(descs, 5, 2, 5, 2)
        s["out"] = torch.empty(n_out, dtype=torch.int64, device="cuda")
    return s


def run(s):
    op, B = s["op"], s["batch"]
    if op == "polymul_f64":
        s["plan"].multiply_f64(s["a"], s["b"], s["out"], B)
        return s["out"]
    if op == "polymul_split":
        s["plan"].multiply_i32(s["a"], s["b"], s["out"], B)
        return s["out"]
    if op == "ffnt_product":
        twist, root, untwist, iroot = s["tables"]
        G.GPU_FFNT(s["real"], s["temp"], twist, root, s["fwd"], 2 * B)
        G.GPU_FFNT(s["out"], s["temp"], untwist, iroot, s["inv"], B, True)
        return s["out"]
    if op == "rr_product":
        G.GPU_FFT_R(s["real"], s["temp"], s["tables"][0], s["fwd"], 2 * B)
        G.GPU_FFT_R(s["out"], s["temp"], s["tables"][1], s["inv"], B, True)
        return s["out"]
    if op == "c2c_product":
        # the transforms run in place, so the operands are copied in first
        s["x"].copy_(s["src"])
        G.GPU_FFT(s["x"], s["tables"][0], s["fwd"], 2 * B)
        G.GPU_FFT(s["x"], s["tables"][1], s["inv"], B, True)
        return s["product"]
    if op == "c2c_round":
        G.GPU_FFT(s["x"], s["tables"][0], s["fwd"], B)
        G.GPU_FFT(s["x"], s["tables"][1], s["inv"], B)
        return s["x"]
    if op == "special_round":
        G.GPU_Special_FFT(s["x"], s["tables"][1], s["inv"], B)
        G.GPU_Special_FFT(s["x"], s["tables"][0], s["fwd"], B)
        return s["x"]
    if op == "ckks":
        G.ckks_decode(s["m"], s["slots"], s["tables"][0], s["n"], 2.0 ** 30, B)
        G.ckks_encode(s["slots"], s["coeffs"], s["tables"][1], s["n"], 2.0 ** 30, B, s["work"])
        return s["slots"], s["coeffs"]
    s["plan"].execute(s["a"], s["b"], s["out"])
    return s["out"]


# ---- what a pass cannot do without ----
def _fft_flops(n):
    return 5.0 * n * (1 << n)


def work(case):
    op = case["op"]
    if op == "batched":
        kinds, rings = _list(case)
        nbytes = flops = 0.0
        for k, r in zip(kinds, rings):
            nbytes += 8.0 * (1 << r) + 8.0 * G.output_length(k, r)
            flops += 3 * _fft_flops(r - 1 if k == G.PRODUCT_NEGACYCLIC else r)
        return {"bytes": nbytes, "flops": flops}
    B = case["batch"]
    n = case["ring"] if "ring" in case else case["n"]
    N = 1 << n
    r = 4 if case.get("prec") == "f32" else 8
    c = 2 * r
    if op == "polymul_f64":
        return {"bytes": 24.0 * N * B, "flops": 3 * B * _fft_flops(n - 1)}
    if op == "polymul_split":
        # the function itself: three transforms of doubles would do
        return {"bytes": 16.0 * N * B, "flops": 3 * B * _fft_flops(n - 1)}
    if op == "ffnt_product":
        # two calls: reals to spectra, spectra to reals
        return {"bytes": B * N * (2.0 * r + c + c + r), "flops": 3 * B * _fft_flops(n - 1)}
    if op == "rr_product":
        return {"bytes": B * N * (2.0 * r + 2 * c + 2 * c + r), "flops": 3 * B * _fft_flops(n)}
    if op == "c2c_product":
        return {"bytes": B * N * c * (4.0 + 4.0 + 3.0), "flops": 3 * B * _fft_flops(n)}
    if op in ("c2c_round", "special_round"):
        return {"bytes": 4.0 * B * N * c, "flops": 2 * B * _fft_flops(n)}
    return {"bytes": 4.0 * B * N * 16, "flops": 2 * B * _fft_flops(n)}  # ckks


# ---- the same in 64 bits ----
def _product(a, b, nega):
    """Rows of a times rows of b mod X^N -+ 1, integers, on the host."""
    a, b = a.double().cpu(), b.double().cpu()
    N = a.shape[-1]
    full = torch.fft.irfft(torch.fft.rfft(a, 2 * N) * torch.fft.rfft(b, 2 * N), 2 * N)
    full = torch.round(full)
    return full[..., :N] - full[..., N:] if nega else full[..., :N] + full[..., N:]


def exact(case, seed):
    op = case["op"]
    if op in ("c2c_round", "special_round"):
        return _signal(case, seed).to(torch.complex128).cpu()
    if op == "ckks":
        n, B = case["n"], case["batch"]
        l, N = 1 << n, 2 << n
        m = _coeffs(case, seed).cpu()
        z = m.view(B, N).double() * torch.exp(1j * math.pi / N * torch.arange(N, dtype=torch.float64))
        values = torch.fft.ifft(z, norm="forward")  # m at zeta^(2k + 1)
        k = [1] * l
        for j in range(1, l):
            k[j] = 5 * k[j - 1] % (2 * N)
        at = (torch.tensor(k) - 1) // 2
        return (values[:, at] / 2.0 ** 30).reshape(-1), m
    a, b = _operands(case, seed)
    if op == "batched":
        kinds, rings = _list(case)
        a, b = a.cpu(), b.cpu()
        out, at = [], 0
        for k, r in zip(kinds, rings):
            x, y = a[at:at + (1 << r)], b[at:at + (1 << r)]
            at += 1 << r
            if k == G.PRODUCT_LINEAR:
                pad = torch.zeros_like(x)
                out.append(_product(torch.cat((x, pad)), torch.cat((y, pad)), True))
            else:
                out.append(_product(x, y, True))
        return torch.cat(out).to(torch.int64)
    nega = op not in ("rr_product", "c2c_product") or bool(case.get("nega"))
    p = _product(a.view(case["batch"], -1), b.view(case["batch"], -1), nega).reshape(-1)
    if op == "polymul_split":
        return p.to(torch.int64)
    return p.to(torch.complex128) if op == "c2c_product" else p
