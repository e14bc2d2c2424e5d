"""A plan that runs its two inner dimensions as planes reports that: the
description names the launches, and the pass times and bytes are those of the two
launches it runs, not of the three passes it does not."""
import ctypes
import time

import numpy as np
import pytest

import pfft_amd as P
from gpu_util import spec_of, random_input, run_gpu, oracle_out, rel_l2
from test_gpu_timer import timer_vec
from shared_comm import shared_comm   # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


def times(plan, a, b, iters=20):
    L = P.lib()
    L.pfft_amd_plan_npasses.argtypes = [ctypes.c_void_p]
    L.pfft_amd_time_passes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                       ctypes.c_int, ctypes.POINTER(ctypes.c_double),
                                       ctypes.POINTER(ctypes.c_double)]
    k = L.pfft_amd_plan_npasses(plan.handle)
    ms, by = (ctypes.c_double * k)(), (ctypes.c_double * k)()
    assert L.pfft_amd_time_passes(plan.handle, a.ptr, b.ptr, iters, ms, by) == 0
    return list(ms), list(by)


@pytest.mark.parametrize("flags", [0, P.TRANSPOSED_OUT])
def test_reports_the_launches(flags):
    n = [2048, 64, 64]
    size = 16 * n[0] * n[1] * n[2]
    rc, comm = P.create_procmesh([1, 1])
    a, b = P.DeviceBuffer(size), P.DeviceBuffer(size)
    plan = P.Plan("c2c", n, a.ptr, b.ptr, comm=comm, flags=flags | P.ESTIMATE)
    lines = plan.describe()
    assert len(lines) == 3
    planes = [ln for ln in lines if ":plane " in ln]
    assert len(planes) == 2 and all(" launch=" in ln for ln in lines), lines
    ms, by = times(plan, a, b)
    assert len(ms) == 3 and sum(by) == 4 * size   # two sweeps, each read and written
    plan.execute()
    best = 1e9
    for _ in range(20):
        t0 = time.perf_counter()
        plan.execute()
        best = min(best, 1e3 * (time.perf_counter() - t0))
    print("passes %s ms, execution %.4f ms" % (["%.4f" % v for v in ms], best))
    # two sweeps of 268 MB at 5 TB/s, 0.1 ms, and 0.012 ms of events, against an
    # execution that holds both launches and 0.01 ms of host work; three passes
    # take half as much again
    assert sum(ms) < 1.2 * best
    plan.destroy()
    a.free()
    b.free()


def test_last_plane_counts_its_last_round():
    # 600 planes on 512 workgroups: the second round has 88; a round of 512 planes
    # of 64 KiB takes 12 us and more, a late one of 88 half that and more; events
    # hold 6 us beside them: 18 / 24 of the interval, 12 / 24 without the second round
    n = [600, 64, 64]
    size = 16 * n[0] * n[1] * n[2]
    rc, comm = P.create_procmesh([1, 1])
    a, b = P.DeviceBuffer(size), P.DeviceBuffer(size)
    plan = P.Plan("c2c", n, a.ptr, b.ptr, comm=comm, flags=P.ESTIMATE)
    lines = plan.describe()
    ms, _ = times(plan, a, b)
    ev = sum(t for t, ln in zip(ms, lines) if ":plane " in ln)
    L = P.lib()
    L.pfft_reset_timer.argtypes = [ctypes.c_void_p]
    L.pfft_reset_timer(plan.handle)
    for _ in range(20):
        plan.execute()
    r, v = timer_vec(plan)
    got = 1e3 * (v[5] + v[6]) / v[3]   # dimensions 2 and 1: trafo[0], trafo[1]
    print("planes: timer %.4f ms, events %.4f ms" % (got, ev))
    assert 0.62 * ev < got < 1.15 * ev
    plan.destroy()
    a.free()
    b.free()


@pytest.mark.parametrize("prec,n", [("f64", [1100, 60, 64]), ("f32", [4700, 20, 21])])
@pytest.mark.parametrize("flags", [0, P.TRANSPOSED_OUT])
def test_second_plane_of_a_workgroup(prec, n, flags):
    # more planes than resident workgroups (16 waves a CU of at least a wave each:
    # 4096 at most, 512 of 60x64 complex128): the tables are kept for the next plane
    spec = spec_of("c2c", n, flags=flags)
    x = random_input(spec, 3)
    y = run_gpu(spec, x, prec=prec, plan_flags_extra=P.ESTIMATE)
    assert rel_l2(y, oracle_out(spec, x)) < (1e-12 if prec == "f64" else 2e-6)
