"""GPU: the pair cache while single vertices move far.  Vertices that moved a
quarter of the skin or more are listed, and they and the vertices with one of
them among their candidates take the full query; more than 32 in a block of 256
or 256 in all record every list again.  Energy, gradient and per-vertex
properties equal those of the full query bit for bit on every step: the move
itself, evaluations with the vertices out there, small moves of all between
(some cross a cell), the way back, and flips and rebuilds in between."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_pair_cache import core, pair, same    # noqa: F401

pytestmark = pytest.mark.gpu


def patch(x, at, count):
    """The count vertices nearest to vertex at (in few blocks of the library's
    spatial order)."""
    return np.argsort(((x - x[at]) ** 2).sum(axis=1))[:count]


@pytest.mark.parametrize("excl", [0, 1, 2])
@pytest.mark.parametrize("count,together", [(1, 1), (3, 0), (20, 1), (32, 1), (33, 1), (60, 1), (40, 0), (255, 0),
                                            (300, 0), (700, 0)])
def test_far_moves_of_some(core, excl, count, together):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(4, seed=7)
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, excl, "mixed")
    rng = np.random.default_rng(count)
    same(mesh, on, off, "start")
    for step in range(3):
        x = mesh.points()
        some = patch(x, int(rng.integers(len(x))), count) if together else rng.choice(len(x), count, replace=False)
        move = rng.normal(0.0, 0.5 * lbar, (count, 3))
        x[some] += move
        same(mesh, on, off, "out")
        for k in range(3):
            x[:] = x + rng.normal(0.0, 0.006 * lbar, x.shape)
            same(mesh, on, off, f"out there {k}")
        x[some[:count // 2]] -= move[:count // 2]
        same(mesh, on, off, "half of them back")
        x[some[count // 2:]] -= move[count // 2:]
        same(mesh, on, off, "all back")
        if step == 0:
            # uniforms of zero accept every flip that the topology allows
            edges = rng.permutation(mesh.n_edges())[:200].astype(np.int32)
            assert core.flip_injected(mesh, on, edges, np.zeros(200))[0] > 0
        elif step == 1:
            on.update_repulsion(mesh)
            off.update_repulsion(mesh)
        same(mesh, on, off, "after")


def test_positions_that_are_not_numbers(core):    # noqa: F811
    """A trajectory that overflowed: NaN and infinite rows count as fast, and
    the lists of the others stay right after they are gone."""
    v, f, lbar = M.jittered_icosphere(3, seed=8)
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, 0, "mixed")
    same(mesh, on, off, "start")
    for bad in (np.nan, np.inf, -np.inf, 1e300):
        x = mesh.points().copy()
        mesh.points()[17] = bad
        a, b = on.energy(mesh), off.energy(mesh)
        assert a == b or (np.isnan(a) and np.isnan(b))
        assert np.array_equal(on.gradient(mesh), off.gradient(mesh), equal_nan=True)
        mesh.points()[:] = x
        same(mesh, on, off, "back")
