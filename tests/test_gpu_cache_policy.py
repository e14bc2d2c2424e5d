"""Passes over arrays of 16 to 288 MiB leave their intermediates in the
memory-side cache (cache_policy in plan.c), which the power-of-two kernels
run as instantiations of their own: parity with the oracle over their
lengths, kinds, lane orders, ragged tiles, embeds and shifts."""
import pytest

import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, out_mask, rel_l2

pytestmark = pytest.mark.gpu

TI, TO = P.TRANSPOSED_IN, P.TRANSPOSED_OUT
SH = P.SHIFTED_IN | P.SHIFTED_OUT

CASES = [
    ("c2c", [130, 64, 150], None, 0, "f64"),
    ("c2c", [128, 75, 130], None, TO, "f64"),
    ("c2c", [256, 65, 70], None, TI, "f64"),
    ("c2c", [512, 50, 45], None, 0, "f64"),
    ("c2c", [9, 1024, 128], None, 0, "f64"),
    ("c2c", [5, 2048, 105], None, 0, "f64"),
    ("c2c", [3, 4096, 90], None, 0, "f64"),
    ("r2c", [129, 64, 256], None, TO, "f64"),
    ("c2r", [129, 64, 256], None, TI, "f64"),
    ("c2c", [128, 160, 128], None, TO, "f32"),
    ("c2c", [3, 512, 1400], None, 0, "f32"),
    ("r2c", [130, 128, 256], None, TO, "f32"),
    ("c2r", [130, 128, 256], None, TI, "f32"),
    ("r2c", [128, 128, 256], [100, 90, 200], SH, "f32"),
]


@pytest.mark.parametrize("extra", [0, P.ESTIMATE])
@pytest.mark.parametrize("kind,n,ni,flags,prec", CASES)
def test_kept_intermediates_parity(kind, n, ni, flags, prec, extra):
    spec = spec_of(kind, n, ni, sign=(+1 if kind == "c2r" else -1), flags=flags)
    x = random_input(spec, 3)
    y = run_gpu(spec, x, prec=prec, plan_flags_extra=extra)
    assert rel_l2(y, oracle_out(spec, x), out_mask(spec)) < (1e-12 if prec == "f64" else 2e-6)
