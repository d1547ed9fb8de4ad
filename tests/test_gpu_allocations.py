"""GPU: what a step with the caller's momenta needs on the device is there before it
(a step allocates nothing: its thread may have another device current, and its
stream may be recording)."""
import ctypes

import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_replicas import core, params    # noqa: F401

pytestmark = pytest.mark.gpu


def free_bytes():
    h = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert h.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_steps_with_momenta_allocate_nothing(core):    # noqa: F811
    """16 meshes of 40962 vertices, whose rows are 16 MB together: enough to show
    in the free memory, which is given out in larger blocks."""
    v, f, lbar = M.jittered_icosphere(6, seed=5)
    chains = []
    for _ in range(17):
        mesh = core.TriMesh(v, f)
        est = core.EnergyManager(mesh, params(core, lbar))
        est.gradient(mesh)
        chains.append((mesh, est, core.DeviceHMC(mesh, est)))
    p = np.random.default_rng(1).normal(size=v.shape)
    kw = dict(mass=1.0, time_step=1e-5, num_integration_steps=2, temperature=1.0, momenta=p, uniform=0.5)
    chains[0][2].step(**kw)    # brings in what the process allocates once
    before = free_bytes()
    for c in chains[1:]:
        c[2].step(**kw)
    assert free_bytes() == before
