"""r2r lines in one launch where there are few of them: a plan of floats moves half
the bytes of one of doubles through the same launches and takes no longer; parity
at the line counts where the tile width changes."""
import time

import pytest

import gpu_util
import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, rel_l2
from test_gpu_mixed import KINDS
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


def plan_us(n, kind, prec, howmany):
    size = howmany * 8
    for v in n:
        size *= v
    a, b = P.DeviceBuffer(size), P.DeviceBuffer(size)
    plan = P.Plan("r2r", n, a.ptr, b.ptr, howmany=howmany, comm=gpu_util.comm_for(1), prec=prec,
                  kinds=[KINDS[kind]] * len(n), flags=P.ESTIMATE)
    assert plan.ok
    best = 1e9
    for _ in range(60):
        t0 = time.perf_counter()
        plan.execute()
        best = min(best, time.perf_counter() - t0)
    plan.destroy()
    a.free()
    b.free()
    return 1e6 * best


@pytest.mark.parametrize("kind", ["DHT", "REDFT10", "REDFT01", "REDFT11", "RODFT11"])
@pytest.mark.parametrize("n,howmany", [([1024, 128], 2), ([128, 128, 8], 1), ([64, 64, 16], 1),
                                       ([64, 64, 3], 1)])
def test_floats_no_slower_than_doubles(n, howmany, kind):
    f32, f64 = plan_us(n, kind, "f32", howmany), plan_us(n, kind, "f64", howmany)
    print(n, howmany, kind, "floats %.1f us, doubles %.1f us" % (f32, f64))
    assert f32 < 1.1 * f64   # 1.1 for the clock


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("n", [[5, 100, 411], [5, 101, 819], [9, 64, 1820], [3, 100, 3], [2, 130, 1]])
def test_line_counts(n, kind, prec):
    # 2055 and 4095 lines across memory, 16380, 9 and 2
    kinds = [KINDS[kind] if d == 1 else P.DHT for d in range(3)]
    n = list(n)
    n[1] += {"REDFT00": 1, "RODFT00": -1}.get(kind, 0) if n[1] % 2 == 0 else 0
    spec = spec_of("r2r", n, kinds=kinds)
    x = random_input(spec, 4)
    assert rel_l2(run_gpu(spec, x, prec=prec), oracle_out(spec, x)) < (1e-12 if prec == "f64" else 4e-6)
