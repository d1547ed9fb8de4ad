"""GPU: loss and parameter gradient on a topology that flips have changed since the
network was made, against autograd on the CPU restatement."""
import numpy as np
import pytest
import torch

import surrogate_ref as S

from test_gpu_surrogate import core, randomize, ref_inputs, system    # noqa: F401

pytestmark = pytest.mark.gpu


def test_backward_follows_the_flips(core):    # noqa: F811
    v, f, mesh, est, om, oe = system(core, 2, seed=9)
    est.precision = "fp64"
    sg = core.Surrogate(mesh, est, seed=2)
    randomize(sg, 5)
    prop = np.random.default_rng(3).choice(mesh.n_edges(), 24, replace=False).astype(np.int32)
    uni = np.zeros(24)
    acc = core.flip_injected(mesh, est, prop, uni)
    assert acc == oe.flip_serial_injected(om, prop, uni) and acc[0] > 10
    assert np.array_equal(mesh.fv_indices(), om.fv_indices())
    loss, grad = sg.loss_grad()
    fe, sp, nu, sF = ref_inputs(sg, v, om.fv_indices(), om, oe)
    th = torch.tensor(np.asarray(sg.params), requires_grad=True)
    L = S.loss(S.forward(th, fe, sp, nu, sF), oe.gradient(om), sF)
    (ref,) = torch.autograd.grad(L, th)
    ref = ref.numpy()
    # operands rounded to bf16 (2^-9 each) in four products one after another;
    # of a block of the gradient on its own twice that
    assert abs(loss - float(L)) <= 8 * 2.0 ** -9 * float(L)
    rel = np.linalg.norm(grad - ref) / np.linalg.norm(ref)
    print("gradient", rel, flush=True)
    assert rel <= 8 * 2.0 ** -9
    for l in range(S.LAYERS):
        a, b = S.OFF[f"E{l}"], S.OFF[f"b{l}"]
        rel = np.linalg.norm(grad[a:b] - ref[a:b]) / np.linalg.norm(ref[a:b])
        print("E", l, rel, flush=True)
        assert rel <= 16 * 2.0 ** -9
