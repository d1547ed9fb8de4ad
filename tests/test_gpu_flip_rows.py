"""GPU: the flip sweeps' rows of one-rings at the lengths where their reading
and rewriting change: eight slots are moved in registers and compared as two
vectors, sixteen are read at once, thirty-two fill a row.  Bipyramids give two
vertices of the wanted valence; every accepted flip moves it by one, so the
sweeps cross the boundary in both directions."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from trimem_amd import capi
from trimem_amd import meshes as M

from test_gpu_parity import bipyramid, props_vec, to_core_params

pytestmark = pytest.mark.gpu

VALENCES = (3, 7, 8, 9, 15, 16, 17, 31)


@pytest.fixture(scope="module")
def core():
    import trimem_amd.core as m
    assert m.device_count() > 0, "no GPU visible"
    return m


def case(n, excl, kr=1.0):
    v, f = bipyramid(n)
    v = v + np.random.default_rng(n).normal(0.0, 0.01, v.shape)
    lbar = M.mean_edge_length(v, f)
    p = O.Params(kappa_b=1.0, kappa_a=1.0, kappa_v=1.0, kappa_c=1.0, kappa_t=1e-3, kappa_r=kr,
                 bond_lc0=1.25 * lbar, bond_lc1=0.75 * lbar, rep_lc1=1.2 * lbar, rep_rlist=1.2 * lbar,
                 rep_exclusion=excl)
    return v, f, p


@pytest.mark.parametrize("n", VALENCES)
@pytest.mark.parametrize("excl,window", [(2, 256), (2, 5), (1, 256), (0, 256)])
def test_serial_rows_follow_the_oracle(core, n, excl, window):
    """Three passes over all edges in random order, about half the uniforms
    accepting anything: accepted counts, uniforms used and faces are the
    oracle's, and so is the energy on the flipped topology."""
    v, f, p = case(n, excl)
    om, gm = O.Mesh(v, f), core.TriMesh(v, f)
    oe, ge = O.EnergyManager(om, p), core.EnergyManager(gm, to_core_params(core, p))
    t = ge.tuning
    t["serial_window"] = window
    ge.tuning = t
    rng = np.random.default_rng(100 + n)
    ne = gm.n_edges()
    prop = np.concatenate([rng.permutation(ne) for _ in range(3)]).astype(np.int32)
    uni = np.where(rng.random(len(prop)) < 0.5, 0.0, rng.random(len(prop)))
    got = core.flip_injected(gm, ge, prop, uni)
    assert got == oe.flip_serial_injected(om, prop, uni) and got[0] > 0
    assert np.array_equal(gm.fv_indices(), om.fv_indices())
    assert abs(ge.energy(gm) - oe.energy(om)) <= 1e-10 * abs(oe.energy(om))


@pytest.mark.parametrize("n", VALENCES)
@pytest.mark.parametrize("batch", [1, 5, 0])
def test_parallel_rows_keep_the_running_state(core, n, batch):
    """Parallel sweeps whose running properties equal those of the final
    topology evaluated afresh (a row, a claim or a patch difference gone wrong
    would show), at exclusion level 0, where the repulsion counts too."""
    v, f, p = case(n, 0, kr=1e-3)
    m = core.TriMesh(v, f)
    e = core.EnergyManager(m, to_core_params(core, p))
    total = 0
    for k in range(4):
        acc = core.pflip(m, e, 1.0, seed=7 * n + k, batch=batch)
        total += acc
        st = (ctypes.c_double * 8)()
        assert capi.lib().tm_energy_pflip_state(ctypes.c_void_p(e._handle()), st) == 0
        assert int(st[7]) == acc
        for s, x in zip(st[:6], props_vec(e.properties(m))):
            assert abs(s - x) <= 1e-10 * abs(x) + 1e-12
    # with three equator vertices, all adjacent, only the three equator edges
    # can flip, and their cost may refuse them all
    assert total > 0 or n == 3
