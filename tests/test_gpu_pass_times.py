"""The pass times of a plan's timer against event timing of the same passes,
where the last pass leaves its workgroups uneven: 300 tiles of a matrix-core
prime (one workgroup per CU, 256 CUs) take two rounds, the second with 44
workgroups.  A round takes 15 us and more, the two 30 or more, and an event
interval holds about 6 us beside the pass: the timer reads at least 30 / 36 of
it, and at most half if it misses the second round."""
import ctypes

import pytest

import pfft_amd as P
from test_gpu_timer import timer_vec

pytestmark = pytest.mark.gpu


def event_ms(plan, a, b):
    L = P.lib()
    L.pfft_amd_plan_npasses.argtypes = [ctypes.c_void_p]
    L.pfft_amd_time_passes.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                       ctypes.c_int, ctypes.POINTER(ctypes.c_double),
                                       ctypes.POINTER(ctypes.c_double)]
    k = L.pfft_amd_plan_npasses(plan.handle)
    ms, by = (ctypes.c_double * k)(), (ctypes.c_double * k)()
    assert L.pfft_amd_time_passes(plan.handle, a.ptr, b.ptr, 20, ms, by) == 0
    return list(ms)


@pytest.mark.parametrize("kind,n,flags,prec,slot", [
    ("c2c", [40, 60, 587], 0, "f64", 0),
    ("c2c", [40, 60, 1181], 0, "f32", 0),
    ("c2r", [40, 60, 587], P.TRANSPOSED_IN, "f64", 5),
    ("c2r", [40, 60, 1181], P.TRANSPOSED_IN, "f32", 5),
])
def test_last_pass_counts_its_last_round(kind, n, flags, prec, slot):
    rc, comm = P.create_procmesh([1, 1])
    size = 16 * n[0] * n[1] * (n[2] + 1)
    a, b = P.DeviceBuffer(size), P.DeviceBuffer(size)
    plan = P.Plan(kind, n, a.ptr, b.ptr, sign=+1, flags=flags, comm=comm, prec=prec)
    assert plan.ok and plan.describe()[-1].split("kernel=")[-1].startswith("mixed")
    ev = event_ms(plan, a, b)[-1]
    L = P.lib()
    pre = "pfft" if prec == "f64" else "pfftf"
    getattr(L, pre + "_reset_timer").argtypes = [ctypes.c_void_p]
    getattr(L, pre + "_reset_timer")(plan.handle)
    for _ in range(20):
        plan.execute()
    r, v = timer_vec(plan)
    ms = 1e3 * v[5 + slot] / v[3]
    print(kind, n, prec, "timer %.4f ms, events %.4f ms" % (ms, ev))
    assert 0.65 * ev < ms < 1.15 * ev
    plan.destroy()
    a.free()
    b.free()
