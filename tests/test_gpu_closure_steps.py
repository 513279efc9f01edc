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
