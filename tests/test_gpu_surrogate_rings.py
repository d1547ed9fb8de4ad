"""GPU: the surrogate's vertex kernels at the ring lengths where they change
(eight slots of a ring are read together, nine and ten follow; four vertices
share a step, so every remainder of four occurs), against the CPU restatement.
Bipyramids give two vertices of the wanted valence."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from trimem_amd import meshes as M
import surrogate_ref as S

from test_gpu_parity import bipyramid
from test_gpu_surrogate import core, core_params, pdict, randomize, ref_inputs, stages_ref    # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 5, 7, 8, 9, 10])
def test_forward_and_backward_at_every_ring_length(core, n):    # noqa: F811
    v, f = bipyramid(n)
    v = v + np.random.default_rng(n).normal(0.0, 0.03, v.shape)
    d = pdict(M.mean_edge_length(v, f))
    mesh = core.TriMesh(v, f)
    est = core.EnergyManager(mesh, core_params(core, d))
    est.precision = "fp64"
    om = O.Mesh(v, f)
    oe = O.EnergyManager(om, O.Params(**d))
    sg = core.Surrogate(mesh, est, seed=1)
    randomize(sg, n)
    F = sg.forces()
    fe, sp, nu, sF = ref_inputs(sg, v, f, om, oe)
    # sums in another order (2e-5), and some of the 64 N operands of a product
    # rounded to the other neighbour in bf16: four of them at half a unit of
    # 2^-8 against the norm of all
    tol = 2e-5 + 4 * 2.0 ** -9 / np.sqrt(64 * len(v))
    for which, r in enumerate(stages_ref(np.asarray(sg.params), fe, sp, nu)):
        e = np.linalg.norm(sg.activations(which) - r) / np.linalg.norm(r)
        print(n, "stage", which, e, tol, flush=True)
        assert e <= tol
    Fr = S.forward(torch.tensor(np.asarray(sg.params)), fe, sp, nu, sF).numpy()
    assert np.linalg.norm(F - Fr) <= 2 * tol * np.linalg.norm(Fr)
    loss, grad = sg.loss_grad()
    th = torch.tensor(np.asarray(sg.params), requires_grad=True)
    L = S.loss(S.forward(th, fe, sp, nu, sF), oe.gradient(om), sF)
    (ref,) = torch.autograd.grad(L, th)
    assert abs(loss - float(L)) <= 6 * tol * float(L)
    # operands rounded to bf16 (2^-9 each) in four products one after another
    rel = np.linalg.norm(grad - ref.numpy()) / np.linalg.norm(ref.numpy())
    print(n, "gradient", rel, flush=True)
    assert rel <= 8 * 2.0 ** -9
