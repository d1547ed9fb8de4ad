"""GPU: faces read several times after sweeps, on both sides of the size up to which
the second reading brings the topology to the host, and between sweeps that accept
something and sweeps that only swap ids (flip and flip back)."""
import numpy as np
import pytest

from oracle import oracle as O

from test_gpu_parity import core, flip_case, to_core_params    # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [2, 4, 5])    # 320, 5120 and 20480 faces
def test_faces_read_again(core, level):    # noqa: F811
    v, f, p = flip_case(level, 41, False)
    om, gm = O.Mesh(v, f), core.TriMesh(v, f)
    oe, ge = O.EnergyManager(om, p), core.EnergyManager(gm, to_core_params(core, p))
    rng = np.random.default_rng(level)
    for reads, u in ((1, 0.0), (3, 2.0), (2, 0.0), (0, 2.0), (3, 0.0), (3, 2.0)):
        prop = rng.integers(0, gm.n_edges(), 20).astype(np.int32)
        uni = np.full(20, u)
        assert core.flip_injected(gm, ge, prop, uni) == oe.flip_serial_injected(om, prop, uni)
        for _ in range(reads):
            assert np.array_equal(gm.fv_indices(), om.fv_indices())
    assert np.array_equal(gm.fv_indices(), om.fv_indices())
