"""The planner's effort and the wisdom cache reach the launches of a plan that can
run its inner dimensions as planes: planes or one pass per dimension is a timed
selection, and the pass beside the planes takes its own one; every forced
selection runs (its name stands in the description) and computes the
transform."""
import pytest

import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, rel_l2
from test_gpu_tune import _plan_lines, tune_all   # noqa: F401 (fixture)
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu
TO, TI = P.TRANSPOSED_OUT, P.TRANSPOSED_IN


def force(path, plane, other):
    """every selection of the file to `other`, those of planes to `plane`"""
    lines = open(path).read().splitlines()
    out = [lines[0]]
    for ln in lines[1:]:
        key, v, r, ms = ln.split()
        out.append("%s %d %d %s" % ((key,) + (plane if ".q" in key else other) + (ms,)))
    open(path, "w").write("\n".join(out) + "\n")


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("flags", [0, TO, TI])
@pytest.mark.parametrize("n,other,name", [
    ([256, 16, 20], (0, 1), "fast+xcd"), ([256, 16, 20], (2, 0), "fast-narrow"),
    ([256, 16, 20], (4, 1), "fast-grid+xcd"), ([256, 16, 20], (1, 0), "general"),
    ([210, 14, 20], (9, 1), "mixed+xcd"), ([210, 14, 20], (9, 0), "mixed"),
])
def test_forced(tune_all, tmp_path, n, other, name, flags, prec):   # noqa: F811
    t0 = P.tune_timings()
    spec, first = _plan_lines("c2c", n, flags, prec)
    assert P.tune_timings() > t0
    w = tmp_path / "w.txt"
    assert P.export_wisdom(str(w)) == 0
    assert sum(".q" in ln for ln in open(w)) == 1
    tol = 1e-12 if prec == "f64" else 2e-6
    x = random_input(spec, 5)
    ref = oracle_out(spec, x)
    for plane in ((9, 0), (0, 0)):
        force(str(w), plane, other)
        P.forget_wisdom()
        assert P.import_wisdom(str(w)) == 0
        t1 = P.tune_timings()
        _, lines = _plan_lines("c2c", n, flags, prec)
        # the pass beside the planes is timed once if the first plan did not need it
        assert P.tune_timings() == t1
        launches = {ln.split(" launch=")[1].split()[0].split(":")[1] for ln in lines
                    if " launch=" in ln}
        assert launches == ({"plane", name} if plane[0] == 9 else set()), lines
        assert rel_l2(run_gpu(spec, x, prec=prec), ref) < tol


def test_estimate_and_small_plans_keep_the_rule(monkeypatch):
    monkeypatch.delenv("PFFT_AMD_TUNE", raising=False)
    P.forget_wisdom()
    t0 = P.tune_timings()
    for flags in (0, P.ESTIMATE):
        _, lines = _plan_lines("c2c", [256, 16, 20], flags, "f64")
        assert all(" launch=" in ln for ln in lines), lines
    assert P.tune_timings() == t0


def test_large_plan_times_both(monkeypatch, tmp_path):
    monkeypatch.delenv("PFFT_AMD_TUNE", raising=False)
    monkeypatch.delenv("PFFT_AMD_WISDOM", raising=False)
    P.forget_wisdom()
    _plan_lines("c2c", [1024, 32, 48], 0, "f64")
    w = tmp_path / "w.txt"
    assert P.export_wisdom(str(w)) == 0
    assert sum(".q48:" not in ln and ".q32:" in ln for ln in open(w)) == 1
    P.forget_wisdom()
