"""GPU: the pair cache while vertices stay far from where they were recorded: after
twelve evaluations in a row with fast vertices, or an accepted trajectory that ends
with some, all lists are recorded again.  Everything equals the full query bit for
bit before, at and after it: evaluations, device HMC without list rebuilds, and a
replica group's steps."""
import numpy as np
import pytest

from trimem_amd import meshes as M

from test_gpu_pair_cache import core, pair, params, same    # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("excl", [0, 2])
@pytest.mark.parametrize("level", [3, 6])    # sums by the pass itself and by a launch
def test_a_vertex_that_stays_away(core, level, excl):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(level, seed=17)
    mesh = core.TriMesh(v, f)
    on, off = pair(core, mesh, lbar, excl, "mixed")
    rng = np.random.default_rng(4)
    same(mesh, on, off, "start")
    for k in range(20):
        x = mesh.points()
        if k in (1, 16):
            x[rng.integers(len(x), size=3)] += rng.normal(0.0, 0.5 * lbar, (3, 3))
        x[:] = x + rng.normal(0.0, 0.002 * lbar, x.shape)
        same(mesh, on, off, f"step {k}")    # an energy and a gradient and the properties: three evaluations


def test_trajectories_that_drift(core):    # noqa: F811
    v, f, lbar = M.jittered_icosphere(4, seed=18)
    runs = []
    for cache in (1, 0):
        mesh = core.TriMesh(v, f)
        est = core.EnergyManager(mesh, params(core, lbar, 1))
        est.precision = "mixed"
        t = est.tuning
        t["pair_cache"] = cache
        est.tuning = t
        d = core.DeviceHMC(mesh, est)
        out = []
        for s in range(16):    # momenta of 1: a few hundredths of an edge per trajectory
            d.step(mass=1.0, time_step=3e-4, num_integration_steps=10, temperature=1.0, seed=9, step=s)
            r = d.result()
            out.append((r["accepted"], r["dh"], r["energy1"]))
        moved = np.linalg.norm(mesh.points() - v, axis=1).max()
        print("cache", cache, [o[0] for o in out], "largest move / lc1", moved / (1.5 * lbar), flush=True)
        assert moved > 0.05 * 1.5 * lbar    # beyond what a slow vertex moves
        runs.append((mesh.points().copy(), out))
    assert np.array_equal(runs[0][0], runs[1][0])
    assert runs[0][1] == runs[1][1]
    assert any(o[0] for o in runs[0][1])


def test_groups_that_drift(core):    # noqa: F811
    runs = []
    for cache in (1, 0):
        meshes, ests = [], []
        for i, level in enumerate((3, 4, 3)):
            v, f, lbar = M.jittered_icosphere(level, seed=30 + i)
            meshes.append(core.TriMesh(v, f))
            ests.append(core.EnergyManager(meshes[-1], params(core, lbar, 1)))
            ests[-1].precision = "mixed"
        group = core.Replicas(meshes, ests)
        t = group.tuning
        t["pair_cache"] = cache
        group.tuning = t
        group.hmc_setup(mass=1.0, time_step=3e-4, temperature=1.0, seeds=[1, 2, 3], num_integration_steps=10)
        group.hmc_run(16)
        st = group.stats()
        runs.append((np.concatenate([m.points() for m in meshes]), np.asarray(st["props"]), list(st["accepted"])))
        print("cache", cache, runs[-1][2], flush=True)
    assert np.array_equal(runs[0][0], runs[1][0])
    assert np.array_equal(runs[0][1], runs[1][1])
    assert runs[0][2] == runs[1][2] and sum(runs[0][2]) > 0
