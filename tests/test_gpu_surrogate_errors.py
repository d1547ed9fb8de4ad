"""GPU: a loss and gradient that fails leaves the caller's arrays as they were."""
import ctypes

import numpy as np
import pytest

from trimem_amd import capi
from trimem_amd import meshes as M

from test_gpu_parity import bipyramid, max_valence
from test_gpu_surrogate import core, core_params, pdict    # noqa: F401

pytestmark = pytest.mark.gpu


def test_refused_loss_grad_stores_nothing(core):    # noqa: F811
    v, f = bipyramid(10)
    v = v + np.random.default_rng(1).normal(0.0, 0.03, v.shape)
    p = pdict(M.mean_edge_length(v, f))
    # an equator edge: its flip joins the apexes, of valence 10
    for e in range(3 * len(f) // 2):
        mesh = core.TriMesh(v, f)
        est = core.EnergyManager(mesh, core_params(core, p))
        core.flip_injected(mesh, est, np.array([e], np.int32), np.array([0.0]))
        if max_valence(mesh.fv_indices(), len(v)) == 11:
            break
    mesh = core.TriMesh(v, f)
    est = core.EnergyManager(mesh, core_params(core, p))
    lib = capi.lib()
    sg, n = ctypes.c_void_p(), ctypes.c_int()
    assert lib.tm_surrogate_create(ctypes.c_void_p(mesh._handle()), ctypes.c_void_p(est._handle()),
                                   ctypes.c_uint64(1), ctypes.byref(sg)) == 0
    assert lib.tm_surrogate_params(sg, None, ctypes.byref(n)) == 0
    assert core.flip_injected(mesh, est, np.array([e], np.int32), np.array([0.0])) == (1, 1)
    assert max_valence(mesh.fv_indices(), len(v)) == 11
    loss = ctypes.c_double(-7.0)
    grad = np.full(n.value, -7.0, np.float32)
    status = lib.tm_surrogate_loss_grad(sg, ctypes.byref(loss), grad.ctypes.data_as(ctypes.POINTER(ctypes.c_float)))
    lib.tm_surrogate_destroy(sg)
    assert status != 0
    assert loss.value == -7.0 and np.all(grad == -7.0)
