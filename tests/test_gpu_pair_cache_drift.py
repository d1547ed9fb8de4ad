"""GPU: the pair cache while vertices drift across cell boundaries.  Recordings of
small meshes mark the vertices that have no candidate in any cell they can reach
before the next recording, and those keep replaying nothing in whichever of them
they are.  Uniform drifts take many vertices across, in every direction, on
meshes whose sheets nearly touch (candidates just beyond the cells searched) and
on both sides of the size up to which marks are made.  Energy, gradient and
per-vertex properties equal those of the full query bit for bit."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_pair_cache import core, pair, same    # noqa: F401

pytestmark = pytest.mark.gpu


def drift(core, v, f, lbar, excl, rc, seed):    # noqa: F811
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, excl, "mixed", rc)
    rng = np.random.default_rng(seed)
    same(mesh, on, off, "start")
    step = 0.24 * 0.2 * rc * lbar / 3    # three of them stay below the limit, the fourth records
    for k in range(9):
        if k % 3 == 0:
            way = rng.normal(0.0, 1.0, 3)
            way *= step / np.linalg.norm(way)
        x = mesh.points()
        x[:] = x + way + rng.normal(0.0, 0.02 * step, x.shape)
        same(mesh, on, off, f"drift {k}")
    on.update_repulsion(mesh)
    off.update_repulsion(mesh)
    same(mesh, on, off, "rebuilt")


@pytest.mark.parametrize("flat", [1.0, 0.12, 0.05])
@pytest.mark.parametrize("excl", [0, 1, 2])
@pytest.mark.parametrize("rc", [0.8, 1.5, 2.5])
def test_drift_across_cells(core, rc, excl, flat):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(4, seed=13)
    drift(core, v * np.array([1.0, 1.0, flat]), f, lbar, excl, rc, 3)


@pytest.mark.parametrize("rows", [128, 129])
def test_at_the_largest_marked_mesh(core, rows):    # noqa: F811
    """16384 vertices and 128 more, a flattened tube."""
    v, f = M.tube(length=(rows - 0.5) * 2 * np.pi / 128, radius=1.0, segments=128)
    assert len(v) == 128 * rows
    drift(core, v * np.array([1.0, 1.0, 0.05]), f, M.mean_edge_length(v, f), 2, 1.5, 4)
