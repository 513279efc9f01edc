"""ClosureModel.train runs whole epochs in lbm355_closure_train_epoch: per minibatch the gradient (four wavefronts per
block over tiles of 64 samples, summed in a fixed order) and an Adam step."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _setup(n, seed=3):
    from lbmpy_amd.closure import ClosureModel
    m = ClosureModel(seed=seed, nu_scale=1e-3)
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, 10, generator=g).cuda()
    y = torch.rand(n, generator=g).cuda() * 2
    return m, x, y


# one sample, edges of a tile, of a block (256) and of a block's last wavefront, more tiles than wavefronts (131072)
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1000, 131072, 131073 + 64 * 5])
def test_gradient_equals_atomic_sums(n):
    from lbmpy_amd import _native as nat
    m, x, y = _setup(n)
    loss, grad = m.gradient(x, y)
    g2, l2 = torch.empty_like(grad), torch.empty_like(loss)
    p = (lambda t: ctypes.c_void_p(t.data_ptr()))
    nat.check(m.lib.lbm355_closure_train_step(p(m.params), p(x), p(y), n, p(g2), p(l2), 1024,
                                              nat.current_stream_handle()))
    # the same products in another order of FP32 sums: n terms of one sign at worst
    tol = 4 * np.finfo(np.float32).eps * np.sqrt(n) + 1e-6
    assert float((grad - g2).norm() / g2.norm()) <= tol
    assert abs(float(loss - l2)) <= tol * float(l2)
    again = m.gradient(x, y)
    assert torch.equal(again[1], grad) and torch.equal(again[0], loss)


@pytest.mark.parametrize("n,batch", [(1, 7), (300, 64), (1000, 333), (2048, 4096), (140000, 135000)])
def test_epoch_equals_its_steps(n, batch):
    m, x, y = _setup(n)
    r, _, _ = _setup(n)
    history = m.train(x, y, epochs=2, batch=batch, lr=1e-3, seed=5)
    gen = torch.Generator(device=r.device).manual_seed(5)
    want = []
    for _ in range(2):
        perm = torch.randperm(n, generator=gen, device=r.device)
        losses = []
        for s in range(0, n, batch):
            idx = perm[s:s + batch]
            loss, grad = r.gradient(x[idx], y[idx])
            r.adam_step(grad, lr=1e-3)
            losses.append(float(loss[0]))
        want.append(sum(losses) / len(losses))
    assert torch.equal(m.master, r.master) and torch.equal(m.m, r.m) and torch.equal(m.v, r.v)
    assert torch.equal(m.params, r.params) and m.step == r.step
    np.testing.assert_allclose(history, want, rtol=1e-12)


def test_bad_samples_are_refused():
    m, x, y = _setup(64)
    with pytest.raises(ValueError):
        m.train(x.cpu(), y)
    with pytest.raises(ValueError):
        m.train(x[:, :9], y)
    with pytest.raises(ValueError):
        m.train(x, y[:60])
