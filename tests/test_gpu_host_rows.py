"""GPU: rows between host memory and the device at the sizes where their way
changes: an odd number of doubles, one piece of the staging ring (21845 rows of
three doubles, 10922 of six, 43690 faces) and one more, more pieces than the
ring holds, both sides of the size from which positions go through the copy
engine."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_replicas import core, params, vertex_properties    # noqa: F401

pytestmark = pytest.mark.gpu


def strip(n, seed):
    """n vertices in a zigzag: a folded strip of triangles off the origin (its
    volume and curvature, which the energy divides by, are not zero)."""
    i = np.arange(n)
    rng = np.random.default_rng(seed)
    v = np.stack([0.5 * i, (i % 2) * 0.8, 1.0 + 0.3 * (i % 3)], axis=1) + rng.normal(0.0, 0.02, (n, 3))
    k = np.arange(n - 2)
    f = np.where((k % 2 == 0)[:, None], np.stack([k, k + 1, k + 2], 1), np.stack([k + 1, k, k + 2], 1))
    return v, f.astype(np.int32)


@pytest.mark.parametrize("n", [4, 5, 6, 511, 10922, 10923, 21845, 21846, 65535, 65536, 174763])
def test_rows_come_and_go_unchanged(core, n):    # noqa: F811
    """Vertices in random order; every row's energy terms depend on its own
    neighbourhood, so a row that came or went wrong shows.  Positions: up,
    and down again after the host's copy was overwritten."""
    from trimem_amd import capi
    v, f = strip(n, n)
    order = np.random.default_rng(n + 1).permutation(n)
    back = np.argsort(order)
    p = params(core, 1.0, kappa_r=0.0)
    plain, mixed = core.TriMesh(v, f), core.TriMesh(v[order], back[f].astype(np.int32))
    e0, e1 = core.EnergyManager(plain, p), core.EnergyManager(mixed, p)
    for step in range(2):
        rows0, rows1 = vertex_properties(plain, e0), vertex_properties(mixed, e1)
        g0, g1 = e0.gradient(plain), e1.gradient(mixed)
        # the walk round a vertex may start elsewhere: a few roundings per term
        assert np.all(np.abs(rows1 - rows0[order]) <= 1e-12 * np.abs(rows0).max(axis=0))
        assert np.abs(g1 - g0[order]).max() <= 1e-9 * np.abs(g0).max()
        d = capi.lib()
        x = mixed.points().copy()
        assert d.tm_mesh_upload_points(mixed._handle()) == 0
        mixed.points()[:] = 0.0
        assert d.tm_mesh_download_points(mixed._handle()) == 0
        assert np.array_equal(mixed.points(), x)
        shift = np.random.default_rng(step).normal(0.0, 0.01, v.shape)
        plain.points()[:] = v + shift
        mixed.points()[:] = (v + shift)[order]


def test_faces_of_more_than_a_piece(core):    # noqa: F811
    """43690 faces fit a piece; the faces after flips are those of a fresh
    mesh with that connectivity."""
    v, f, lbar = M.jittered_icosphere(6, seed=3)
    mesh = core.TriMesh(v, f)
    est = core.EnergyManager(mesh, params(core, lbar, kappa_r=0.0))
    assert core.pflip(mesh, est, 0.2, seed=1) > 0
    faces = mesh.fv_indices()
    again = core.TriMesh(mesh.points(), faces)
    p = est.properties(mesh)
    q = core.EnergyManager(again, params(core, lbar, kappa_r=0.0)).properties(again)
    assert again.n_faces() == len(f) and again.n_edges() == mesh.n_edges()
    for k in ("area", "volume", "curvature", "bending", "tethering"):
        assert abs(getattr(p, k) - getattr(q, k)) <= 1e-9 * max(1.0, abs(getattr(q, k))), k
