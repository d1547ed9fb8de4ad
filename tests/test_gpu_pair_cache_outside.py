"""GPU: replay of the pair cache for vertices outside the cell grid.  The grid
covers the vertices as they were when the list was built; a vertex that has
left it has a cell there as well, whose candidates it replays.  Energy, gradient
and per-vertex properties equal those of the full query bit for bit, on every
side of the grid, one cell away and beyond its reach."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_pair_cache import core, pair, same    # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("excl", [0, 2])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("cells", [-3.0, -1.2, -0.4, 0.4, 1.2, 3.0])
def test_moved_off_the_grid(core, axis, cells, excl):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(3, seed=9)
    v = v + 5.0    # the grid starts at the origin in y and z: all six sides have cells of the mesh or none
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, excl, "mixed")
    rng = np.random.default_rng(axis)
    same(mesh, on, off, "start")
    for scale in (1.0, 1.1):    # a move of all, then parts that leave on every side
        x = mesh.points()
        mid = x.mean(axis=0)
        shift = np.zeros(3)
        shift[axis] = cells * 1.5 * lbar
        x[:] = mid + (x - mid) * scale + (shift if scale == 1.0 else 0.0)
        same(mesh, on, off, "moved: recorded")
        for k in range(3):
            x[:] = x + rng.normal(0.0, 0.004 * lbar, x.shape)
            same(mesh, on, off, f"replayed {k}")
