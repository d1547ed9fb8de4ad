"""GPU: replays of the pair cache for every number of recorded candidates: none,
up to four (one vector), up to eight (two) and more than eight in a lane (the
full query every time), by the cutoff.  Energy, gradient and per-vertex
properties equal those of the full query bit for bit."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_pair_cache import core, pair, same    # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("excl", [0, 1])
@pytest.mark.parametrize("rc", [0.9, 1.5, 2.2, 3.0, 4.5])
def test_replay_of_every_count(core, rc, excl, precision):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(3, seed=11)
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, excl, precision, rc)
    rng = np.random.default_rng(5)
    total = same(mesh, on, off, "start")[:, 5].sum()
    for k in range(4):
        x = mesh.points()
        x[:] = x + rng.normal(0.0, 0.004 * lbar, x.shape)
        total += same(mesh, on, off, f"replayed {k}")[:, 5].sum()
    assert total > 0 or rc < 1.0 or (excl == 1 and rc < 2.0)
