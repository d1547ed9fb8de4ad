"""GPU: the members of a replica group.  A mesh and its manager may be members more
than once, a mesh may be a member with several managers, meshes without
vertices may stand anywhere among the others, and one member's list may have so many
cells that the scan of the tiles is a launch of its own: each member's results are
those of its mesh alone."""
import ctypes

import numpy as np
import pytest

from trimem_amd import capi
from trimem_amd import meshes as M

from test_gpu_nlist_build import to_core_params
from test_gpu_replicas import core, params    # noqa: F401
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def sphere(core, level, seed, **kw):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(level, seed=seed)
    mesh = core.TriMesh(v, f)
    return mesh, core.EnergyManager(mesh, params(core, lbar, **kw))


def far_spheres(core, cells=204):    # noqa: F811
    """Two small spheres in opposite corners of cells^3 cells: 2073 tiles of them."""
    v, f, _ = M.jittered_icosphere(2, seed=3)
    r = 0.45 / cells
    x = np.concatenate([r * v + r, r * v + (1.0 - r)])
    x -= x.min(axis=0)
    faces = np.concatenate([f, f + len(v)]).astype(np.int32)
    rl = x.max() / (cells + 0.5)
    mesh = core.TriMesh(x, faces)
    p = O.Params(rep_rlist=rl, rep_lc1=rl, rep_exclusion=1, bond_lc0=rl, bond_lc1=0.1 * rl)
    return mesh, core.EnergyManager(mesh, to_core_params(core, p))


def compare(core, group, singles):    # noqa: F811
    group.eval()
    g = group.globals()
    for i, (n, e) in enumerate(singles):
        if n.n_vertices() == 0:
            assert np.all(g[i, :6] == 0.0) and np.isnan(g[i, 6])    # (A / A0 - 1)^2 of 0 / 0
            continue
        assert g[i, 6] == e.energy(n), i
        assert np.array_equal(group.gradient(i), e.gradient(n)), i


@pytest.mark.parametrize("order", [(0, 0), (0, 0, 1), (1, 0, 2, 0, 0, 1)])
@pytest.mark.parametrize("level", [2, 4, 6])
def test_members_again(core, level, order):    # noqa: F811
    """Lists rebuilt and evaluations of a group in which managers come again, at
    sizes whose sums are the pass's own last step (up to 128 blocks) and a
    launch of their own (160)."""
    def members():
        out = [sphere(core, level, 3, excl=1), sphere(core, 3, 4), sphere(core, 3, 5, n_search="verlet-list")]
        return [out[i] for i in order]
    a, b = members(), members()
    group = core.Replicas([m for m, _ in a], [e for _, e in a])
    rng = np.random.default_rng(level)
    for step in range(4):
        done = []
        for (m, _), (n, e) in zip(a, b):
            if n in done:
                continue
            done.append(n)
            move = rng.normal(0.0, (0.02, 0.002)[step % 2], m.points().shape)
            m.points()[:] += move
            n.points()[:] += move
            if step % 2 == 0:
                e.update_repulsion(n)
        if step % 2 == 0:
            group.update_repulsion()
        else:
            for m, _ in a:
                assert capi.lib().tm_mesh_upload_points(ctypes.c_void_p(m._handle())) == 0
        compare(core, group, b)


def test_one_mesh_with_several_managers(core):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(3, seed=8)
    kinds = [dict(excl=1), dict(excl=2, kappa_b=7.0), dict(n_search="verlet-list")]
    m, n = core.TriMesh(v, f), core.TriMesh(v, f)
    a = [core.EnergyManager(m, params(core, lbar, **k)) for k in kinds]
    b = [core.EnergyManager(n, params(core, lbar, **k)) for k in kinds]
    group = core.Replicas([m] * 3, a)
    group.update_repulsion()
    for e in b:
        e.update_repulsion(n)
    compare(core, group, [(n, e) for e in b])


@pytest.mark.parametrize("same_manager", [True, False])
def test_sweeps_of_one_mesh_follow_each_other(core, same_manager):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(4, seed=9)
    m, n = core.TriMesh(v, f), core.TriMesh(v, f)
    ea = core.EnergyManager(m, params(core, lbar))
    other = ea if same_manager else core.EnergyManager(m, params(core, lbar, kappa_b=3.0))
    eb = core.EnergyManager(n, params(core, lbar))
    last = eb if same_manager else core.EnergyManager(n, params(core, lbar, kappa_b=3.0))
    extra, extra1 = sphere(core, 3, 10), sphere(core, 3, 10)
    group = core.Replicas([m, extra[0], m], [ea, extra[1], other])
    acc = group.pflip(0.2, [5, 6, 7])
    want = [core.pflip(n, eb, 0.2, seed=5), core.pflip(extra1[0], extra1[1], 0.2, seed=6),
            core.pflip(n, last, 0.2, seed=7)]
    assert list(acc) == want and min(want) > 0
    assert np.array_equal(m.fv_indices(), n.fv_indices())
    assert np.array_equal(extra[0].fv_indices(), extra1[0].fv_indices())


def test_members_without_vertices_and_with_many_cells(core):    # noqa: F811
    def members():
        def none():
            mesh = core.TriMesh(np.zeros((0, 3)), np.zeros((0, 3), np.int32))
            return mesh, core.EnergyManager(mesh, params(core, 1.0))
        return [none(), sphere(core, 2, 1), none(), none(), far_spheres(core),
                sphere(core, 3, 2, n_search="verlet-list"), none()]
    a, b = members(), members()
    group = core.Replicas([m for m, _ in a], [e for _, e in a])
    compare(core, group, b)
    group.update_repulsion()
    for n, e in b:
        e.update_repulsion(n)
    compare(core, group, b)
    compare(core, group, b)
