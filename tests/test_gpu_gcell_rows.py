"""Blocks of single floats of 16 MiB and more go by the row kernels, blocks of 80
MiB and more through the streaming forms: bitwise the oracle's results at row
widths around the wave and the unrolled span and for ghost widths beyond one
period."""
import pytest

import pfft_amd as P
from test_gpu_gcell import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["exchange", "reduce"])
@pytest.mark.parametrize("n,gb,ga", [
    ([260, 260, 63], [1, 1, 0], [0, 1, 1]), ([1030, 64, 64], [0, 0, 0], [1, 0, 0]),
    ([128, 512, 65], [2, 1, 3], [1, 2, 70]), ([64, 1000, 70], [3, 4, 150], [5, 1, 80]),
    ([64, 65, 1024], [1, 0, 4], [0, 1, 5]), ([4200, 1, 1030], [1, 1, 7], [1, 1, 2]),
])
def test_rows(n, gb, ga, op):
    run("r", n, gb, ga, prec="f32", op=op)


@pytest.mark.parametrize("op", ["exchange", "reduce"])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_streamed_block(prec, op):
    run("r", [128, 820, 200], [2, 1, 3], [1, 2, 2], prec=prec, op=op)
