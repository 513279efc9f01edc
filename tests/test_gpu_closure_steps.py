"""ClosureModel.gradient with a bound on its wavefronts, and more samples than wavefronts take at once, against the CPU
oracle with the tolerances of tests/test_gpu_closure.py (the backward pass rounds its deltas to BF16)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


class _Recorder:
    """A library that notes the calls of its training functions."""

    def __init__(self, lib):
        self.lib, self.calls = lib, []

    def __getattr__(self, name):
        f = getattr(self.lib, name)
        if not name.startswith("lbm355_closure"):
            return f

        def call(*args):
            self.calls.append((name, args))
            return f(*args)
        return call


def _setup(n, seed=3):
    from lbmpy_amd.closure import ClosureModel
    m = ClosureModel(seed=seed, nu_scale=2e-3)
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, 10, generator=g).cuda()
    y = (torch.rand(n, generator=g) * 2).cuda()
    m.lib = _Recorder(m.lib)
    return m, x, y


@pytest.mark.parametrize("n,blocks", [(20000, 97), (5000, 1), (140000, 1024), (300000, 4096)])
def test_gradient_against_the_oracle(n, blocks):
    from oracle import closure_oracle as co
    m, x, y = _setup(n)
    loss, grad = m.gradient(x, y, blocks=blocks)
    (name, args), = [c for c in m.lib.calls if "workspace" not in c[0]]
    if blocks < 1024:
        assert name == "lbm355_closure_train_step" and args[6] == blocks
    else:
        assert name == "lbm355_closure_gradient"
    lo, go = co.loss_and_grad(m.master.cpu().numpy(), m.in_shift, m.in_scale, x.cpu().numpy(), y.cpu().numpy())
    assert abs(float(loss[0]) - lo) <= 1e-3 * lo
    g = grad.cpu().numpy()
    for a, b in ((co.OFF_W1T, co.OFF_W2T), (co.OFF_W2T, co.OFF_W3), (co.OFF_W3, co.OFF_B1), (co.OFF_B1, co.OFF_B2),
                 (co.OFF_B2, co.OFF_B3), (co.OFF_B3, co.MASTER_SIZE)):
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 3e-2 * np.linalg.norm(go[a:b])


def test_training_goes_through_a_models_own_steps():
    from lbmpy_amd.closure import ClosureModel
    seen = []

    class Clipped(ClosureModel):
        def gradient(self, features, targets, blocks=1024):
            loss, grad = super().gradient(features, targets, blocks)
            seen.append(len(features))
            return loss, grad * 0.5

    class Scheduled(ClosureModel):
        def adam_step(self, grad, lr=1e-3, **kw):
            super().adam_step(grad, lr=0.0, **kw)

    _, x, y = _setup(1000)
    plain, clipped, scheduled = (c(seed=3, nu_scale=2e-3) for c in (ClosureModel, Clipped, Scheduled))
    start = scheduled.master.clone()
    for m in (plain, clipped, scheduled):
        assert len(m.train(x, y, epochs=2, batch=300, lr=1e-2)) == 2
        assert m.step == 8
    assert seen == [300, 300, 300, 100] * 2
    assert torch.equal(scheduled.master, start)
    # a gradient of half the size moves Adam's first moment by half, its second by a quarter
    by_hand = ClosureModel(seed=3, nu_scale=2e-3)
    gen = torch.Generator(device="cuda").manual_seed(0)
    for _ in range(2):
        perm = torch.randperm(1000, generator=gen, device="cuda")
        for s in range(0, 1000, 300):
            _, grad = by_hand.gradient(x[perm[s:s + 300]], y[perm[s:s + 300]])
            by_hand.adam_step(grad * 0.5, lr=1e-2)
    assert torch.equal(clipped.master, by_hand.master) and not torch.equal(clipped.master, plain.master)


def test_targets_for_every_sample():
    m, x, _ = _setup(64)
    with pytest.raises(ValueError):
        m.train(x, torch.zeros(32, 2, device="cuda"))


@pytest.mark.parametrize("form", ["float64", "columns", "float16 targets"])
def test_training_converts_no_more_than_its_bound(form):
    """Samples that need a copy, and more of them than the bound, are converted by minibatches, with the same result."""
    from lbmpy_amd.closure import ClosureModel
    n = 200000
    _, x, y = _setup(n)
    y = y.half().float()
    xs, ys = (x.double(), y) if form == "float64" else (x.t().contiguous().t(), y) if form == "columns" else (x, y.half())
    plain, whole, bounded = (ClosureModel(seed=3, nu_scale=2e-3) for _ in range(3))
    for m in (whole, bounded):
        m.lib = _Recorder(m.lib)
    bounded.MOST_CONVERTED = 4 * ys.numel() - 1
    plain.train(x, y, epochs=1, batch=30000)
    for m in (whole, bounded):
        m.train(xs, ys, epochs=1, batch=30000)
        assert torch.equal(plain.master, m.master) and plain.step == m.step
    assert [c[0] for c in whole.lib.calls if "workspace" not in c[0]] == ["lbm355_closure_train_epoch"]
    sizes = [c[1][3] for c in bounded.lib.calls if c[0] == "lbm355_closure_gradient"]
    assert sizes == [30000] * 6 + [20000] and not any("epoch" in c[0] for c in bounded.lib.calls)
