"""The mixed-radix kernel (mixed_tile.hpp): parity with the oracle over its
radices (codelets and matrix-core primes), stage counts, tile remainders and every form a pass can take (real
and complex, contiguous, strided and transposing sides, embed / trunc /
shifts, interleaved tuples, in place, adjoint weights)."""
import re

import numpy as np
import pytest

import pfft_amd as P
from oracle import layout as L
from gpu_util import (spec_of, random_input, run_gpu, oracle_out, out_mask, rel_l2, comm_for,
                      n_scalars)

pytestmark = pytest.mark.gpu

TI, TO, PAD = P.TRANSPOSED_IN, P.TRANSPOSED_OUT, P.PADDED_R2C
SH = P.SHIFTED_IN | P.SHIFTED_OUT
TOL = {"f64": 1e-12, "f32": 2e-6}

# lengths by radix list: one codelet, two and three stages, every codelet
LENGTHS = [7, 9, 11, 13, 14, 18, 21, 22, 26, 28, 33, 35, 42, 63, 70, 77, 91, 110, 130, 156, 165,
           176, 182, 196, 210, 225, 250, 300, 360, 495, 500, 1001, 1331, 2197, 4000,
           17, 19, 23, 29, 31, 34, 37, 58, 61, 62, 67, 93, 97, 127, 128 * 3, 157, 251, 289, 323, 510]


def run(kind, n, ni=None, no=None, flags=0, howmany=1, prec="f64", **kw):
    spec = spec_of(kind, n, ni, no, howmany, sign=(+1 if kind == "c2r" else -1), flags=flags)
    x = random_input(spec, 11)
    y = run_gpu(spec, x, prec=prec, **kw)
    assert rel_l2(y, oracle_out(spec, x), out_mask(spec)) < TOL[prec]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths(n, prec):
    # strided, then contiguous lines, with a ragged last tile
    run("c2c", [3, n, 11], prec=prec)
    run("c2c", [3, 5, n], flags=TO, prec=prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [7, 14, 21, 22, 26, 28, 33, 35, 70, 98, 165, 196, 250, 330, 420, 715,
                               17, 31, 34, 62, 74, 97, 106, 127, 254, 289])
@pytest.mark.parametrize("kind,flags", [("r2c", TO), ("r2c", PAD), ("c2r", TI), ("c2r", PAD)])
def test_real_lines(kind, flags, n, prec):
    run(kind, [5, 7, n], flags=flags, prec=prec)


@pytest.mark.parametrize("kind,flags", [("c2c", TO), ("c2c", TI), ("r2c", 0), ("c2r", 0)])
@pytest.mark.parametrize("howmany", [2, 3])
def test_tuples(kind, flags, howmany):
    run(kind, [21, 14, 22], flags=flags, howmany=howmany)


@pytest.mark.parametrize("flags", [0, SH, P.SHIFTED_IN, P.SHIFTED_OUT])
@pytest.mark.parametrize("kind", ["c2c", "r2c", "c2r"])
def test_embed_trunc_shift(kind, flags):
    run(kind, [42, 22, 70], [30, 14, 52], [26, 18, 40], flags=flags)
    run(kind, [42, 22, 70], [30, 14, 52], [26, 18, 40], flags=flags, prec="f32")


@pytest.mark.parametrize("kind", ["r2c", "c2r"])
def test_odd_real_embed(kind):
    run(kind, [9, 7, 35], [5, 7, 21], [9, 5, 27])
    run(kind, [19, 7, 37], [11, 7, 21], [19, 5, 27])


@pytest.mark.parametrize("kind", ["c2c", "r2c", "c2r"])
def test_prime_embed_shift(kind):
    run(kind, [34, 38, 58], [20, 38, 30], [34, 22, 40], flags=SH)


def test_in_place():
    run("c2c", [33, 42, 35], inplace=True)
    run("r2c", [33, 42, 70], flags=PAD, inplace=True)


@pytest.mark.parametrize("n", [31, 35, 62, 70])
@pytest.mark.parametrize("kind", ["c2c", "r2c", "c2r"])
def test_adjoint_dot(kind, n):
    # <A x, y> = <x, A^T y> in the real inner product
    spec = spec_of(kind, [6, 21, n], sign=(+1 if kind == "c2r" else -1))
    x = random_input(spec, 1)
    y = np.random.default_rng(2).uniform(-1, 1, n_scalars(spec, "out"))
    lhs = np.dot(run_gpu(spec, x), y)
    rhs = np.dot(x, run_gpu(spec, y, adjoint=True))
    assert abs(lhs - rhs) < 1e-12 * np.linalg.norm(x) * np.linalg.norm(y) * 6 * 21 * n


def test_named():
    a = P.DeviceBuffer(16 * 210 * 196 * 4)
    pl = P.Plan("c2c", [210, 196, 4], a.ptr, a.ptr, comm=comm_for(2))
    names = [ln.split("kernel=")[-1] for ln in pl.describe()]
    pl.destroy()
    assert names.count("mixed") == 2, names


# ---- r2r lines as one launch (even inner length) ----
KINDS = {"DHT": P.DHT, "REDFT00": P.REDFT00, "REDFT01": P.REDFT01, "REDFT10": P.REDFT10,
         "REDFT11": P.REDFT11, "RODFT00": P.RODFT00, "RODFT01": P.RODFT01,
         "RODFT10": P.RODFT10, "RODFT11": P.RODFT11}
# even lengths with codelet and matrix-core inner lengths; the 00 kinds have the
# inner lengths n - 1 and n + 1, of any parity
R2R_LENGTHS = [8, 10, 14, 18, 22, 34, 62, 64, 100, 128, 250, 256, 640, 1100]
R2R_ODD = [9, 13, 17, 33, 65, 129]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_r2r_lines(kind, prec):
    for n in R2R_LENGTHS + (R2R_ODD if kind.endswith("00") else []):
        # strided lines on a ragged tile, then contiguous ones
        for shape in ([3, n, 19], [3, 5, n]):
            spec = spec_of("r2r", shape, kinds=[P.DHT if d != shape.index(n) else KINDS[kind]
                                                for d in range(3)])
            x = random_input(spec, 5)
            y = run_gpu(spec, x, prec=prec)
            assert rel_l2(y, oracle_out(spec, x)) < (1e-12 if prec == "f64" else 4e-6), shape


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_r2r_embed_tuple_transposed(kind):
    spec = spec_of("r2r", [14, 22, 18], [10, 16, 18], [14, 12, 10], kinds=[KINDS[kind]] * 3,
                   howmany=2, flags=TO)
    x = random_input(spec, 6)
    assert rel_l2(run_gpu(spec, x), oracle_out(spec, x)) < 1e-12


def test_r2r_named():
    a = P.DeviceBuffer(8 * 64 * 64 * 64)
    pl = P.Plan("r2r", [64, 64, 64], a.ptr, a.ptr, comm=comm_for(2), kinds=[P.REDFT10] * 3)
    assert all(ln.endswith("kernel=r2r-mixed") for ln in pl.describe()), pl.describe()
    pl.destroy()
