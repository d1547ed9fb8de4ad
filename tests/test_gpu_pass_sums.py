"""GPU: the global sums of a properties pass on both sides of the row count
(128 rows of 256 vertices) up to which the pass's last workgroup forms them."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_replicas import core, params, vertex_properties    # noqa: F401

pytestmark = pytest.mark.gpu

# one row, 8 rows full and just passed, 128 rows nearly full (32500 vertices),
# 136 rows (33000), a large remainder
SEGMENTS = ((20, 3), (64, 32), (64, 33), (250, 130), (250, 132), (300, 150))


def system(core, segments, rows, precision, seed, **kw):
    v, f = M.tube(length=(rows - 0.5) * 2 * np.pi / segments, radius=1.0, segments=segments)
    v = v + np.random.default_rng(seed).normal(0.0, 0.01 * 2 * np.pi / segments, v.shape)
    mesh = core.TriMesh(v, f)
    assert mesh.n_vertices() == segments * rows
    est = core.EnergyManager(mesh, params(core, M.mean_edge_length(v, f), **kw))
    est.precision = precision
    return mesh, est


@pytest.mark.parametrize("segments,rows", SEGMENTS)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kw", [{}, {"n_search": "verlet-list", "excl": 1}, {"kappa_r": 0.0}])
def test_globals_are_the_sums_of_the_rows(core, segments, rows, precision, kw):    # noqa: F811
    mesh, est = system(core, segments, rows, precision, rows, **kw)
    for k in range(3):
        rows_ = vertex_properties(mesh, est)
        p = est.properties(mesh)
        got = np.array([p.area, p.volume, p.curvature, p.bending, p.tethering, p.repulsion])
        # two orders of adding N terms differ by at most 2 N rounding errors
        # of the absolute sum
        bound = 2 * len(rows_) * np.finfo(float).eps * np.abs(rows_).sum(axis=0)
        assert np.all(np.abs(got - rows_.sum(axis=0)) <= bound), (k, got, rows_.sum(axis=0))
        mesh.points()[:] *= 1.0 + 1e-4


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_group_of_both_kinds_equals_the_meshes(core, precision):    # noqa: F811
    reps = [system(core, s, r, precision, 10 + i, **kw) for i, (s, r, kw) in enumerate(
        [(64, 33, {}), (250, 132, {}), (20, 3, {"kappa_r": 0.0}), (250, 130, {"excl": 1}),
         (250, 132, {"kappa_r": 0.0}), (64, 32, {"n_search": "verlet-list", "excl": 1})])]
    group = core.Replicas([m for m, _ in reps], [e for _, e in reps])
    for k in range(3):
        group.eval()
        g = group.globals()
        for i, (m, e) in enumerate(reps):
            assert g[i, 6] == e.energy(m), (k, i)
            p = e.properties(m)
            assert list(g[i, :6]) == [p.area, p.volume, p.curvature, p.bending, p.tethering, p.repulsion], (k, i)
