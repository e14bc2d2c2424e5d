"""Plane passes (plane_tile.hpp): the two inner dimensions of a 3-d complex
transform in one launch where a plane fits LDS.  Parity with the oracle over
row and column radices, chunked stages, the layouts, both precisions and
directions, in place and the adjoint.  A plan by itself takes the plane pass
from 192 planes on, the plans of a batch from 1024 planes in all (with a
filler plan here)."""
import numpy as np
import pytest

import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, rel_l2, comm_for, n_scalars

pytestmark = pytest.mark.gpu

TI, TO = P.TRANSPOSED_IN, P.TRANSPOSED_OUT
TOL = {"f64": 1e-12, "f32": 2e-6}
FILLER = spec_of("c2c", [1024, 2, 3])

# one to three stages a side, every codelet radix, up to the LDS limit (110
# KiB) and beyond it (the three-pass form), sides with primes above 13
PLANES = [(2, 2), (3, 16), (16, 3), (5, 7), (8, 9), (10, 11), (12, 13), (14, 15), (24, 32), (30, 18),
          (64, 64), (48, 100), (7, 900), (900, 7), (2, 700), (80, 81), (121, 50), (96, 96), (17, 20),
          (110, 112), (128, 128)]


def run_batch(specs, prec, calls=1):
    rdt = np.float64 if prec == "f64" else np.float32
    work = []
    for i, spec in enumerate(specs):
        x = random_input(spec, 20 + i)
        a, b = (P.DeviceBuffer(x.size * np.dtype(rdt).itemsize) for _ in range(2))
        a.upload(x.astype(rdt))
        pl = P.Plan("c2c", spec.n, a.ptr, b.ptr, sign=spec.sign, flags=spec.flags,
                    comm=comm_for(spec.rnk_pm), prec=prec)
        assert pl.ok
        work.append((spec, x, a, b, pl))
    for _ in range(calls):
        P.execute_batch([w[4] for w in work])
        for spec, x, a, b, pl in work:
            y = b.download(rdt, x.size).astype(np.float64)
            assert rel_l2(y, oracle_out(spec, x)) < TOL[prec], (spec.n, spec.sign, spec.flags)
    for w in work:
        w[4].destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n1,n2", PLANES)
def test_planes(n1, n2, prec):
    run_batch([FILLER] + [spec_of("c2c", [5, n1, n2], sign=s, flags=f)
                          for s, f in ((-1, 0), (+1, TO), (-1, TI))], prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_batch_of_all_sizes(prec):
    # launches of every wave count, graph replays
    run_batch([FILLER] + [spec_of("c2c", [3, a, b]) for a, b in PLANES], prec, calls=3)


@pytest.mark.parametrize("n", [[192, 8, 9], [200, 64, 20], [3000, 8, 9], [250, 33, 64]])
@pytest.mark.parametrize("flags", [0, TO, TI])
@pytest.mark.parametrize("rnk_pm", [1, 2])
def test_alone_and_adjoint(n, flags, rnk_pm):
    spec = spec_of("c2c", n, flags=flags, rnk_pm=rnk_pm)
    x = random_input(spec, 3)
    y = run_gpu(spec, x)
    assert rel_l2(y, oracle_out(spec, x)) < 1e-12
    g = np.random.default_rng(4).uniform(-1, 1, n_scalars(spec, "out"))
    lhs, rhs = np.dot(y, g), np.dot(x, run_gpu(spec, g, adjoint=True))
    assert abs(lhs - rhs) < 1e-12 * np.linalg.norm(x) * np.linalg.norm(g) * np.prod(n) ** 0.5


def test_in_place():
    spec = spec_of("c2c", [300, 20, 21])
    x = random_input(spec, 2)
    assert rel_l2(run_gpu(spec, x, inplace=True), oracle_out(spec, x)) < 1e-12
