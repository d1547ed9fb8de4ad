"""GPU: the windowed serial sweep decides as the one-workgroup sweep to the last
bit.  For a proposal in the middle of a sweep the largest uniform that the
one-workgroup sweep accepts is found by bisection over the doubles; the windowed
sweep must accept that one and refuse the next."""
import ctypes
import struct

import numpy as np
import pytest

from oracle import oracle as O
from trimem_amd import meshes as M

from test_gpu_flip_rows import case as rows_case
from test_gpu_parity import core, flip_case, to_core_params    # noqa: F401

pytestmark = pytest.mark.gpu


def bits(x):
    return struct.unpack("<q", struct.pack("<d", x))[0]


def double(b):
    return struct.unpack("<d", struct.pack("<q", b))[0]


def sweep(core, case, w, prop, uni):    # noqa: F811
    v, f, p = case
    m = core.TriMesh(v, f)
    e = core.EnergyManager(m, to_core_params(core, p))
    t = e.tuning
    t["serial_window"] = w
    e.tuning = t
    got = core.flip_injected(m, e, prop, uni)
    return got, m.fv_indices().copy()


def thresholds(core, case, seed, before, sizes=(1, 2, 3, 9, 40, 130, 200, 255)):    # noqa: F811
    """Proposals drawn from few edges, so that the same edges and vertices come
    again within a window; the earlier ones all rejected, or about half of
    them accepted.  The number of proposals whose threshold was compared."""
    ne = core.TriMesh(case[0], case[1]).n_edges()
    rng = np.random.default_rng(seed)
    found = 0
    for n in sizes:
        pool = rng.integers(0, ne, max(4, ne // 8))
        for _ in range(8):
            prop = rng.choice(pool, n).astype(np.int32)
            uni = np.where(rng.random(n) < (0.5 if before == "mixed" else 0.0), 0.0, 2.0)
            uni[-1] = 2.0
            (acc0, used), _ = sweep(core, case, 0, prop, uni)
            if used < 1:
                continue
            # the last valid proposal's uniform is the last one used; those after
            # it, which its flip could make valid, are left out
            while len(prop) > 1 and sweep(core, case, 0, prop[:-1], uni)[0][1] == used:
                prop = prop[:-1]
            uni = uni[:used]
            last = used - 1

            def takes(w, u):
                uni[last] = u
                (acc, _), faces = sweep(core, case, w, prop, uni)
                return acc, faces

            uni[last] = 2.0
            (acc0, _), _ = sweep(core, case, 0, prop, uni)
            if takes(0, 0.5 ** 40)[0] != acc0 + 1 or takes(0, 1.0)[0] != acc0:
                continue    # not flippable, downhill, or too far uphill
            lo, hi = bits(0.5 ** 40), bits(1.0)
            while hi - lo > 1:
                mid = (lo + hi) // 2
                if takes(0, double(mid))[0] == acc0 + 1:
                    lo = mid
                else:
                    hi = mid
            for w in (7, 256):
                for b, acc in ((lo, acc0 + 1), (hi, acc0), (lo - 1, acc0 + 1), (hi + 1, acc0)):
                    a, faces = takes(w, double(b))
                    ref = takes(0, double(b))
                    assert ref[0] == acc
                    assert a == acc, (n, w, double(b))
                    assert np.array_equal(faces, ref[1])
            found += 1
            break
    return found


@pytest.mark.parametrize("level,seed,rep,nlist,excl", [(2, 5, False, 0, 1), (2, 6, True, 0, 0), (3, 7, True, 0, 1),
                                                       (3, 8, True, 0, 2), (3, 9, True, 1, 1)])
@pytest.mark.parametrize("before", ["rejected", "mixed"])
def test_thresholds_to_the_last_bit(core, level, seed, rep, nlist, excl, before):    # noqa: F811
    assert thresholds(core, flip_case(level, seed, rep, nlist, excl), seed, before) >= 4


@pytest.mark.parametrize("n", [9, 17, 31])
@pytest.mark.parametrize("before", ["rejected", "mixed"])
def test_thresholds_of_long_rings(core, n, before):    # noqa: F811
    """Two vertices of valence n, which every patch holds or touches."""
    assert thresholds(core, rows_case(n, 2, kr=1e-3), n, before, (1, 5, 20, 60)) >= 2


@pytest.mark.parametrize("bond", [0, 1])
def test_thresholds_of_an_open_tube(core, bond):    # noqa: F811
    v, f = M.tube(length=1.0, radius=0.5, segments=24)
    lbar = M.mean_edge_length(v, f)
    v = v + np.random.default_rng(3).normal(0, 0.03 * lbar, v.shape)
    p = O.Params(kappa_b=1.0, kappa_a=1.0, kappa_v=1.0, kappa_c=1.0, kappa_t=1.0, kappa_r=1.0, bond_type=bond,
                 bond_a0=0.43 * lbar * lbar, bond_lc0=1.25 * lbar, bond_lc1=0.75 * lbar, rep_lc1=1.5 * lbar,
                 rep_rlist=1.5 * lbar, rep_exclusion=2)
    assert thresholds(core, (v, f, p), 4, "mixed", (1, 5, 40, 130)) >= 2
