"""What tells passes apart in the wisdom cache: the r2r kinds of one line length
share the extended length, but each has a kernel of its own, so each has a
selection of its own; so has a pass whose arrays are kept in the memory-side
cache, beside the same pass in another plan that streams them."""
import pytest

import pfft_amd as P
from gpu_util import comm_for

pytestmark = pytest.mark.gpu


@pytest.fixture
def tune_all(monkeypatch):
    monkeypatch.setenv("PFFT_AMD_TUNE", "2")
    monkeypatch.delenv("PFFT_AMD_WISDOM", raising=False)
    monkeypatch.delenv("PFFT_AMD_XCD_REMAP", raising=False)
    P.forget_wisdom()
    yield
    P.forget_wisdom()


def plan_once(kind, n, prec="f64", **kw):
    size = 16
    for v in n:
        size *= v
    a, b = P.DeviceBuffer(size), P.DeviceBuffer(size)
    p = P.Plan(kind, n, a.ptr, b.ptr, comm=comm_for(2), prec=prec, **kw)
    assert p.ok
    p.destroy()
    a.free()
    b.free()


def test_r2r_kinds_apart(tune_all):
    kinds = [P.REDFT10, P.REDFT01, P.RODFT10, P.RODFT01]   # extended length 4 n
    counts = []
    for k in kinds:
        plan_once("r2r", [10, 14, 22], kinds=[k] * 3)
        counts.append(P.wisdom_count())
    assert counts == [3, 6, 9, 12], counts
    plan_once("r2r", [10, 14, 22], kinds=[P.REDFT01] * 3)
    assert P.wisdom_count() == 12


def test_cache_marks_apart(tune_all, tmp_path):
    # 40 MiB: the user's array is kept; every selection names its marks
    plan_once("c2c", [160, 128, 128])
    f = tmp_path / "w.txt"
    assert P.export_wisdom(str(f)) == 0
    keys = [ln.split()[0] for ln in f.read_text().splitlines()[1:]]
    assert len(keys) == 3 and all(".c3." in k for k in keys), keys
