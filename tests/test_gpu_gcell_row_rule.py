"""Which blocks of single floats go by the row kernels: long rows only, and, with
streamed scratch copies (288 MiB and more), only where that keeps whole
128-byte segments.  An exchange of floats moves half the bytes of one of doubles
and takes no longer than it at any row width; the results are bitwise the
oracle's on both sides of each limit."""
import time

import pytest

import pfft_amd as P
from gpu_util import comm_for
from test_gpu_gcell import run

pytestmark = pytest.mark.gpu


def exchange_us(n, prec):
    box = 1
    for v in n:
        box *= v + 2
    d = P.DeviceBuffer(box * (8 if prec == "f64" else 4))
    plan = P.GcPlan("r", n, d.ptr, [1] * 3, [1] * 3, comm=comm_for(2), prec=prec)
    assert plan.ok
    best = 1e9
    for _ in range(30):
        t0 = time.perf_counter()
        plan.exchange()
        best = min(best, time.perf_counter() - t0)
    plan.destroy()
    d.free()
    return 1e6 * best


@pytest.mark.parametrize("n", [[512, 512, 64], [2000, 70, 70], [400, 400, 100], [300, 300, 192],
                               [300, 200, 286], [128, 256, 512]])
def test_floats_no_slower_than_doubles(n):
    f32, f64 = exchange_us(n, "f32"), exchange_us(n, "f64")
    print(n, "floats %.1f us, doubles %.1f us" % (f32, f64))
    assert f32 < 1.1 * f64   # half the bytes, the same launches; 1.1 for the clock


@pytest.mark.parametrize("op", ["exchange", "reduce"])
@pytest.mark.parametrize("n,gb,ga", [
    ([160, 160, 191], [1, 0, 1], [0, 1, 0]), ([160, 160, 192], [1, 0, 1], [0, 1, 2]),
    ([130, 128, 287], [1, 0, 0], [0, 1, 0]), ([130, 128, 287], [1, 0, 1], [0, 1, 0]),
    ([130, 128, 288], [0, 2, 0], [1, 0, 300]), ([700, 220, 30], [1, 1, 130], [0, 0, 140]),
    # user's array streamed, its copy not (272 MiB of both and more), by rows and linear
    ([200, 400, 500], [1, 0, 6], [0, 1, 6]), ([400, 990, 100], [1, 0, 6], [0, 1, 6]),
    # above 288 MiB: whole segments, ragged rows, ragged boxes
    ([300, 500, 512], [1, 0, 16], [0, 1, 16]), ([300, 500, 512], [1, 0, 1], [0, 1, 1]),
    ([310, 500, 500], [1, 0, 6], [0, 1, 6]),
])
def test_limits_bitwise(n, gb, ga, op):
    run("r", n, gb, ga, prec="f32", op=op)
