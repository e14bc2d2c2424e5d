"""Which plans of a batch run as planes: a batch of many tiny planes takes no
longer than the same transforms with both shifts, which always run as three
short-length passes (the same lines and bytes, signs besides); parity of batches
on both sides of the rule and of tiny planes in plans that run by themselves."""
import time

import numpy as np
import pytest

import gpu_util
import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, rel_l2
from test_gpu_plane import run_batch
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


def batch_us(n, count, prec, flags):
    pts = 2 * n[0] * n[1] * n[2] * (8 if prec == "f64" else 4)
    bufs = [(P.DeviceBuffer(pts), P.DeviceBuffer(pts)) for _ in range(count)]
    comm = gpu_util.comm_for(2)
    plans = [P.Plan("c2c", n, a.ptr, b.ptr, flags=flags, comm=comm, prec=prec) for a, b in bufs]
    assert all(p.ok for p in plans)
    best = 1e9
    for _ in range(20):
        t0 = time.perf_counter()
        P.execute_batch(plans)
        best = min(best, time.perf_counter() - t0)
    for p in plans:
        p.destroy()
    for a, b in bufs:
        a.free()
        b.free()
    return 1e6 * best


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,count", [([1024, 4, 4], 100), ([1000, 2, 2], 40), ([128, 4, 4], 200)])
def test_tiny_planes_no_slower_than_three_passes(n, count, prec):
    plain = batch_us(n, count, prec, 0)
    three = batch_us(n, count, prec, P.SHIFTED_IN | P.SHIFTED_OUT)
    print(n, count, prec, "plain %.1f us, shifted %.1f us" % (plain, three))
    assert plain < 1.15 * three


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,count", [
    ([1100, 2, 2], 3), ([400, 4, 4], 3), ([520, 4, 4], 3), ([700, 7, 9], 9), ([700, 8, 8], 8),
    ([700, 8, 8], 9),
])
def test_batches_at_the_rule(n, count, prec):
    run_batch([spec_of("c2c", n, sign=(-1) ** i) for i in range(count)], prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [[192, 2, 2], [200, 5, 7], [193, 3, 16], [300, 16, 3]])
def test_tiny_planes_alone(n, prec):
    spec = spec_of("c2c", n)
    x = random_input(spec, 3)
    assert rel_l2(run_gpu(spec, x, prec=prec), oracle_out(spec, x)) < (1e-12 if prec == "f64" else 2e-6)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_noalloc_planes_and_tiny_planes(prec):
    # planes of several wave counts and three-pass plans in one fixed work-list,
    # the geometries behind its tasks; a second call with other plans follows
    rdt = np.float64 if prec == "f64" else np.float32
    comm = gpu_util.comm_for(2)
    for sides in ([(64, 64), (4, 4), (20, 30), (16, 16), (7, 9), (96, 80)], [(8, 8), (30, 18)]):
        work = []
        for i in range(24):
            spec = spec_of("c2c", [120, *sides[i % len(sides)]], sign=(-1) ** i)
            x = random_input(spec, i)
            a, b = (P.DeviceBuffer(x.size * np.dtype(rdt).itemsize) for _ in range(2))
            a.upload(x.astype(rdt))
            pl = P.Plan("c2c", spec.n, a.ptr, b.ptr, sign=spec.sign, comm=comm, prec=prec)
            assert pl.ok
            work.append((spec, x, a, b, pl))
        assert P.execute_batch_noalloc([w[4] for w in work]) == 0
        for spec, x, a, b, pl in work[:len(sides)] + work[-len(sides):]:
            y = b.download(rdt, x.size).astype(np.float64)
            assert rel_l2(y, oracle_out(spec, x)) < (1e-12 if prec == "f64" else 2e-6), spec.n
        for w in work:
            w[4].destroy()
