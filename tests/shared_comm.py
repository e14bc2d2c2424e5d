"""A fixture for tests with many plans: one process mesh of each dimension for all
of them (the library registers 4096 meshes in a process)."""
import functools

import pytest

import gpu_util

_made = functools.lru_cache(None)(gpu_util.comm_for)


@pytest.fixture(autouse=True)
def shared_comm(monkeypatch):
    import test_gpu_plane
    import test_gpu_tune
    for mod in (gpu_util, test_gpu_plane, test_gpu_tune):
        monkeypatch.setattr(mod, "comm_for", _made)
