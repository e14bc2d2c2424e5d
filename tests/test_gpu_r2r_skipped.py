"""Skipped dimensions of r2r plans: their arrays are real, so the copying pass moves
single reals (as complex values it reached twice as far as the arrays go, and with
differing layouts moved the wrong ones).  Parity with the oracle over layouts, embeds,
tuples, shifts and both precisions, with nothing written behind the output, alone and
in a batch."""
import numpy as np
import pytest

import gpu_util
import pfft_amd as P
from gpu_util import spec_of, random_input, oracle_out, rel_l2, n_scalars
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu
TI, TO = P.TRANSPOSED_IN, P.TRANSPOSED_OUT
SH = P.SHIFTED_IN | P.SHIFTED_OUT
K = [P.REDFT10, P.RODFT11, P.DHT, P.REDFT01]

CASES = [
    ([26, 32, 2], None, None, 1, TO, 1, [1, 1, 0]),
    ([4, 56, 256], [3, 56, 256], None, 1, 0, 1, [0, 1, 0]),
    ([8, 6, 10], None, None, 1, 0, 2, [0, 1, 0]),
    ([8, 6, 10], None, None, 3, TO, 2, [1, 0, 0]),
    ([12, 14, 10], [8, 10, 6], [12, 12, 8], 2, TI, 2, [0, 0, 1]),
    ([12, 14, 10], [8, 10, 6], [12, 12, 8], 1, SH, 2, [1, 1, 0]),
    ([5, 7, 9, 6], None, None, 1, TO, 2, [1, 0, 1, 0]),
    ([40, 33, 50], None, None, 1, 0, 2, [1, 1, 1]),
]


def plan_and_buffers(case, prec, seed):
    n, ni, no, howmany, flags, rnk_pm, skip = case
    spec = spec_of("r2r", n, ni, no, howmany, 0, flags, rnk_pm, skip, K[:len(n)])
    rdt = np.float64 if prec == "f64" else np.float32
    x = random_input(spec, seed).astype(rdt)
    nin, nout = n_scalars(spec, "in"), n_scalars(spec, "out")
    guard = 4096
    a, b = P.DeviceBuffer(nin * x.itemsize), P.DeviceBuffer((nout + guard) * x.itemsize)
    a.upload(x)
    b.upload(np.full(nout + guard, 7.0, rdt))
    pl = P.Plan("r2r", n, a.ptr, b.ptr, ni, no, howmany, 0, flags, comm=gpu_util.comm_for(rnk_pm),
                skip=skip, prec=prec, kinds=K[:len(n)])
    assert pl.ok
    return spec, x, a, b, pl, nout, rdt


def verify(spec, x, b, nout, rdt, prec):
    y = b.download(rdt)
    assert np.all(y[nout:] == 7.0)
    assert rel_l2(y[:nout].astype(np.float64), oracle_out(spec, x.astype(np.float64))) < \
        (1e-12 if prec == "f64" else 4e-6)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("case", CASES)
def test_skipped(case, prec):
    spec, x, a, b, pl, nout, rdt = plan_and_buffers(case, prec, 3)
    assert any(ln.endswith("kernel=copy") for ln in pl.describe())
    pl.execute()
    verify(spec, x, b, nout, rdt, prec)
    pl.destroy()


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_skipped_in_a_batch(prec):
    # kinds of short lines, which the batch's general kernel runs, beside the copies
    cases = [([5, 7, 6], None, None, 1, TO, 2, [0, 1, 0]), ([4, 3, 7], None, None, 2, 0, 2, [1, 0, 0])]
    work = [plan_and_buffers(c, prec, i) for i, c in enumerate(cases)]
    P.execute_batch([w[4] for w in work])
    for spec, x, a, b, pl, nout, rdt in work:
        verify(spec, x, b, nout, rdt, prec)
        pl.destroy()
