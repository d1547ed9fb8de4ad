"""GPU: building neighbour lists at the sizes where the build changes: one tile
of 4096 cells or vertices and one more, more than 2048 tiles of cells (the scan
of the totals is then a launch of its own), cells of many vertices (more than
the nine rows they share), and the lists of a replica group, built together."""
import numpy as np
import pytest

from oracle import oracle as O
from trimem_amd import meshes as M

from test_gpu_parity import to_core_params
from test_gpu_replicas import core, params    # noqa: F401

pytestmark = pytest.mark.gpu


def check(core, v, f, rl, ltype, step):    # noqa: F811
    p = O.Params(rep_nlist=ltype, rep_rlist=rl, rep_exclusion=1)
    om, gm = O.Mesh(v, f), core.TriMesh(v, f)
    onl, gnl = O.NeighbourList(om, p), core.make_nlist(gm, to_core_params(core, p))
    do, io, jo = onl.distance_matrix(om, rl)
    dg, ig, jg = gnl.distance_matrix(gm, rl)
    assert len(do) > 0
    assert sorted(zip(io.tolist(), jo.tolist(), do.tolist())) == sorted(zip(ig, jg, dg))
    if ltype == 0:
        for pid in range(0, len(v), step):    # candidates in the reference's order
            d0, j0 = onl.point_distances(om, pid, rl)
            assert list(j0) == list(gnl.point_distances(gm, pid, rl)[1])


@pytest.mark.parametrize("ltype", [0, 1])
@pytest.mark.parametrize("cells", [1, 15, 16, 203, 204])
def test_cells_of_every_tile_count(core, cells, ltype):    # noqa: F811
    """Two small spheres in opposite corners of a box of cells^3."""
    v, f, _ = M.jittered_icosphere(2, seed=3)
    side = 1.0
    r = 0.45 / max(cells, 4)
    a, b = r * v + r, r * v + (side - r)
    x = np.concatenate([a, b])
    x -= x.min(axis=0)
    faces = np.concatenate([f, f + len(v)]).astype(np.int32)
    rl = x.max() / (cells + 0.5)
    check(core, x, faces, rl, ltype, 5)


@pytest.mark.parametrize("segments,rows", [(65, 63), (64, 64), (17, 241), (128, 64)])
def test_vertices_at_the_tile(core, segments, rows):    # noqa: F811
    v, f = M.tube(length=(rows - 0.5) * 2 * np.pi / segments, radius=1.0, segments=segments)
    assert len(v) == segments * rows
    v = v + np.random.default_rng(rows).normal(0.0, 0.005, v.shape)
    check(core, v, f, 1.5 * M.mean_edge_length(v, f), 0, 97)


def test_groups_build_what_single_meshes_build(core):    # noqa: F811
    def members():
        out = []
        for i, (level, kw) in enumerate([(2, {}), (4, {"excl": 2}), (3, {"n_search": "verlet-list", "excl": 1}),
                                         (3, {"kappa_r": 0.0}), (4, {"excl": 1}), (2, {"n_search": "verlet-list"})]):
            v, f, lbar = M.jittered_icosphere(level, seed=20 + i)
            if i % 2:
                v = v * np.array([1.0, 1.0, 0.1])
            mesh = core.TriMesh(v, f)
            out.append((mesh, core.EnergyManager(mesh, params(core, lbar, **kw))))
        return out
    a, b = members(), members()
    group = core.Replicas([m for m, _ in a], [e for _, e in a])
    rng = np.random.default_rng(1)
    for step in range(3):
        for (m, _), (n, e) in zip(a, b):
            move = rng.normal(0.0, 0.05, m.points().shape)
            m.points()[:] += move
            n.points()[:] += move
            e.update_repulsion(n)
        group.update_repulsion()
        group.eval()
        g = group.globals()
        for i, (n, e) in enumerate(b):
            assert g[i, 6] == e.energy(n), (step, i)
            assert np.array_equal(group.gradient(i), e.gradient(n)), (step, i)
