"""The mixed-radix kernel where a workgroup takes several tiles, the last one
ragged: LDS and the two sets of line offsets are reused from tile to tile.  Every
case has 1.1 to 6 times as many tiles as the GPU has resident workgroups (256
CUs), for each kind of pass, lines across and along memory, codelet radices and
matrix-core primes.  And every launch form of the kernel, forced through a wisdom
file: variant 9 with the workgroups in order and by XCD."""
import pytest

import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, out_mask, rel_l2
from test_gpu_tune import _plan_lines, _rewrite, tune_all   # noqa: F401 (fixture)
from test_gpu_mixed import KINDS
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu
TI, TO = P.TRANSPOSED_IN, P.TRANSPOSED_OUT


def check(spec, tol64=1e-12, tol32=2e-6, **kw):
    x = random_input(spec, 7)
    ref, mask = oracle_out(spec, x), out_mask(spec)
    for prec, tol in (("f64", tol64), ("f32", tol32)):
        y = run_gpu(spec, x, prec=prec, **kw)
        assert rel_l2(y, ref, mask) < tol, (spec.kind, spec.n, prec)


@pytest.mark.parametrize("n", [[9, 500, 1201], [18, 577, 500], [7, 331, 1201], [6, 1201, 331]])
@pytest.mark.parametrize("sign", [-1, +1])
def test_c2c(n, sign):
    check(spec_of("c2c", n, sign=sign), plan_flags_extra=P.ESTIMATE)


@pytest.mark.parametrize("n", [[20, 577, 840], [20, 577, 675], [6, 1201, 662]])
@pytest.mark.parametrize("kind", ["r2c", "c2r"])
def test_real(kind, n):
    check(spec_of(kind, n, sign=(+1 if kind == "c2r" else -1)), plan_flags_extra=P.ESTIMATE)


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_r2r(kind):
    m, n = {"REDFT00": (29, 151), "RODFT00": (29, 149)}.get(kind, (15, 300))
    for shape, d in (([m, n, 1201], 1), ([m, 1201, n], 2)):
        check(spec_of("r2r", shape, kinds=[KINDS[kind] if k == d else P.DHT for k in range(3)]),
              tol32=4e-6, plan_flags_extra=P.ESTIMATE)


FORCED = [
    ("c2c", [30, 70, 90], TO), ("c2c", [33, 35, 50], TI), ("c2c", [9, 500, 601], 0),
    ("c2c", [64, 128, 256], 0), ("c2c", [14, 37, 62], 0), ("c2c", [21, 300, 700], 0),
    ("r2c", [30, 28, 210], TO), ("r2c", [20, 300, 420], 0), ("r2c", [12, 14, 75], TO),
    ("c2r", [30, 28, 210], TI), ("c2r", [20, 300, 420], 0), ("c2r", [12, 14, 62], TI),
]


@pytest.mark.parametrize("remap", [0, 1])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind,n,flags", FORCED)
def test_forced_variant(tune_all, tmp_path, kind, n, flags, prec, remap):   # noqa: F811
    spec, _ = _plan_lines(kind, n, flags, prec)
    w = tmp_path / "w.txt"
    assert P.export_wisdom(str(w)) == 0
    _rewrite(str(w), 9, remap)
    P.forget_wisdom()
    assert P.import_wisdom(str(w)) == 0
    t0 = P.tune_timings()
    _, lines = _plan_lines(kind, n, flags, prec)
    assert P.tune_timings() == t0
    for ln in lines:   # complex128 lines of a prime length end at 587: two tiles of 8 in LDS
        long_prime = prec == "f64" and " nf=601 " in ln
        want = "general" if long_prime else "mixed" + ("+xcd" if remap else "")
        assert ln.endswith("kernel=" + want), ln
    x = random_input(spec, 5)
    y = run_gpu(spec, x, prec=prec)
    assert rel_l2(y, oracle_out(spec, x), out_mask(spec)) < (1e-12 if prec == "f64" else 2e-6)


@pytest.mark.parametrize("kind", ["REDFT10", "REDFT01", "REDFT11", "DHT"])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_forced_r2r(tune_all, tmp_path, kind, prec):   # noqa: F811
    spec = spec_of("r2r", [10, 60, 700], kinds=[KINDS[kind]] * 3)
    x = random_input(spec, 5)
    ref = oracle_out(spec, x)
    run_gpu(spec, x, prec=prec)   # tunes
    w = tmp_path / "w.txt"
    assert P.export_wisdom(str(w)) == 0
    for remap in (0, 1):
        _rewrite(str(w), 9, remap)
        P.forget_wisdom()
        assert P.import_wisdom(str(w)) == 0
        t0 = P.tune_timings()
        assert rel_l2(run_gpu(spec, x, prec=prec), ref) < (1e-12 if prec == "f64" else 4e-6)
        assert P.tune_timings() == t0
