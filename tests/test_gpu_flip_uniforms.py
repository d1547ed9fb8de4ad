"""GPU: injected uniforms outside [0, 1) and at its ends.  The rule is
u <= min(1, exp(-dE)) (flips.cpp:57-64) at every window size: a negative uniform
accepts, one above 1 or not a number never does."""
import numpy as np
import pytest

from oracle import oracle as O

from test_gpu_parity import core, flip_case, with_window    # noqa: F401

pytestmark = pytest.mark.gpu

INF = float("inf")


@pytest.mark.parametrize("w", [0, 7, 256])
@pytest.mark.parametrize("values", [(2.0,), (-1.0,), (0.0,), (1.0,), (INF,), (-INF,), (float("nan"),),
                                    (2.0, -1.0, 0.0, 1.0, INF, -INF, float("nan"), 0.5)])
def test_uniforms_at_and_outside_the_ends(core, w, values):    # noqa: F811
    v, f, p = flip_case(3, 31, True, 0, 1)
    om, gm = O.Mesh(v, f), core.TriMesh(v, f)
    oe, ge = O.EnergyManager(om, p), with_window(core, gm, p, w)
    rng = np.random.default_rng(8)
    prop = rng.integers(0, gm.n_edges(), gm.n_edges() // 2).astype(np.int32)
    uni = np.asarray(values)[rng.integers(0, len(values), len(prop))]
    got = core.flip_injected(gm, ge, prop, uni)
    assert got == oe.flip_serial_injected(om, prop, uni)
    assert np.array_equal(gm.fv_indices(), om.fv_indices())
    if values in ((2.0,), (INF,)) or values[0] != values[0]:
        assert got[0] == 0
    if values in ((-1.0,), (0.0,), (-INF,)):
        assert got[0] == got[1] > 0
