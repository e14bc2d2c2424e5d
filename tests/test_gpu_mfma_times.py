"""The matrix-core kernels write the clock stamps of a plan's timer: every
pass of the forms has a time, and the passes fit in the wall time of the
execute, for the whole, embedded and shifted lines and the long ones."""
import pytest

import pfft_amd as P
from test_gpu_timer import timer_vec

pytestmark = pytest.mark.gpu
SH = P.SHIFTED_IN | P.SHIFTED_OUT


@pytest.mark.parametrize("form", [P.AMD_MFMA_F32, P.AMD_MFMA_BF16X2])
@pytest.mark.parametrize("n,flags", [
    ([256, 512, 256], 0),
    ([256, 256, 1024], P.ESTIMATE),
    ([256, 32, 512], SH),
    ([2048, 17, 256], 0),
    ([16, 4096, 24], 0),
])
def test_every_pass_has_a_time(form, n, flags):
    rc, comm = P.create_procmesh([1, 1])
    size = 8 * n[0] * n[1] * n[2] * 2
    d_in, d_out = P.DeviceBuffer(size), P.DeviceBuffer(size)
    plan = P.Plan("c2c", n, d_in.ptr, d_out.ptr, sign=-1, flags=flags | form, comm=comm,
                  prec="f32")
    assert plan.ok
    for _ in range(3):
        plan.execute()
    r, v = timer_vec(plan)
    trafo = v[5:5 + 2 * r + 2]
    assert {i for i, x in enumerate(trafo) if x > 0} == {0, 1, 2}, trafo
    assert sum(trafo) <= v[4]
    plan.destroy()
    d_in.free()
    d_out.free()
