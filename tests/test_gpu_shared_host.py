"""GPU: what calls on different meshes share on the host: the staging ring (results
of several pieces asked for by several threads at once) and the list build's tables
(groups of more members than one build takes)."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_replicas import core, params    # noqa: F401

pytestmark = pytest.mark.gpu


def test_results_of_several_threads(core):    # noqa: F811
    from trimem_amd import capi
    lib = capi.lib()
    fn = lib.tm_energy_gradient
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.POINTER(ctypes.c_double)]
    members = []
    for i in range(4):
        v, f, lbar = M.jittered_icosphere(6 if i % 2 else 4, seed=60 + i)    # two pieces and one
        mesh = core.TriMesh(v, f)
        members.append((mesh, core.EnergyManager(mesh, params(core, lbar, kappa_r=0.0))))

    def gradient(i):
        mesh, est = members[i]
        out = np.empty((mesh.n_vertices(), 3))
        assert fn(est._handle(), mesh._handle(), out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))) == 0
        return out

    alone = [gradient(i) for i in range(4)]
    with ThreadPoolExecutor(4) as pool:
        for _ in range(10):
            for i, g in enumerate(pool.map(gradient, range(4))):
                assert np.array_equal(g, alone[i]), i


def test_a_group_of_more_lists_than_one_build(core):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(1, seed=70)
    count, sample = 1030, (0, 1, 1022, 1023, 1024, 1029)
    rng = np.random.default_rng(7)
    xs = [v + rng.normal(0.0, 0.02 * lbar, v.shape) for _ in range(count)]
    meshes = [core.TriMesh(x, f) for x in xs]
    ests = [core.EnergyManager(m, params(core, lbar, excl=i % 3)) for i, m in enumerate(meshes)]
    group = core.Replicas(meshes, ests)
    move = rng.normal(0.0, 0.2 * lbar, v.shape)
    for m in meshes:
        m.points()[:] += move
    group.update_repulsion()
    group.eval()
    g = group.globals()
    for i in sample:
        mesh = core.TriMesh(xs[i], f)
        est = core.EnergyManager(mesh, params(core, lbar, excl=i % 3))
        mesh.points()[:] += move
        est.update_repulsion(mesh)
        assert g[i, 6] == est.energy(mesh), i
