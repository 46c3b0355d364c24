"""tune_polymul times what differs: FP64 plans run one kernel at every radix
setting, FP32-split plans one per radix."""
import pytest

from gpufft_amd import PREC_F32_SPLIT, PREC_F64
from gpufft_amd import autotune as A


class Plan:
    ring_power = 16

    def __init__(self, precision):
        self.precision = precision
        self.radix_bits = 4


@pytest.mark.parametrize("precision,radices", [(PREC_F64, [4]), (PREC_F32_SPLIT, [3, 4, 5])])
def test_candidates(monkeypatch, precision, radices):
    plan, timed = Plan(precision), []
    monkeypatch.setattr(A, "device_key", lambda: "device")
    monkeypatch.setattr(A, "time_ms", lambda run, stream, reps: timed.append(plan.radix_bits) or 1.0)
    cand, ms = A.tune_polymul(plan, lambda: None, None, use_db=False)
    assert timed == radices
    assert plan.radix_bits == cand[0] and sorted(ms) == [(r,) for r in radices]
