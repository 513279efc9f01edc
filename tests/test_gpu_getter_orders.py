"""The macroscopic getter writes FP64 and FP32 fields of any order directly (lbm355_get_fields): x fastest cell by cell,
other orders turned in LDS tiles of 64 cells of x by 16 of the last axis.  Reference: the moments in FP64 from torch."""
import numpy as np
import pytest
import torch

from lbmpy_amd import LBMConfig, LBStencil, create_lb_method, compile_macroscopic_values_getter
from lbmpy_amd.sweep import create_pdf_array

pytestmark = pytest.mark.gpu


def _field(shape, order, dtype):
    """A tensor of `shape` whose axes lie in memory in `order` (slowest first), filled with 7."""
    t = torch.full([shape[a] for a in order], 7.0, dtype=dtype, device="cuda")
    return t.permute(*[order.index(a) for a in range(len(shape))])


# sizes at the edges of the tiles
@pytest.mark.parametrize("size", [(1, 1, 1), (63, 2, 15), (64, 3, 16), (65, 2, 17), (130, 1, 33), (5, 70000 // 350, 3),
                                  (40, 80), (64, 16), (67, 31)])
@pytest.mark.parametrize("order", ["f", "c", "mixed"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("g", [0, 1])
def test_getter_orders(size, order, dtype, g):
    D = len(size)
    st = LBStencil("D2Q9" if D == 2 else "D3Q19")
    m = create_lb_method(LBMConfig(stencil=st, relaxation_rate=1.7, compressible=True, force=(1e-3, 2e-3, 0.0)[:D]))
    rng = np.random.default_rng(1)
    pdf = create_pdf_array(size, st.Q, g, "float64")
    pdf.copy_(torch.from_numpy(0.01 * rng.standard_normal(tuple(pdf.shape))))
    spatial = tuple(pdf.shape[:-1])
    orders = {"f": tuple(range(D - 1, -1, -1)), "c": tuple(range(D)), "mixed": (0,) + tuple(range(D - 1, 0, -1))}[order]
    vorders = {"f": (D,) + orders, "c": orders + (D,), "mixed": orders[:1] + (D,) + orders[1:]}[order]
    rho, dev = (_field(spatial, list(orders), dtype) for _ in range(2))
    u = _field(spatial + (D,), list(vorders), dtype)
    get = compile_macroscopic_values_getter(m, ["density", "density_deviation", "velocity"], ghost_layers=g,
                                            periodicity=(True,) * D)
    get(pdf, density=rho, density_deviation=dev, velocity=u)
    inner = tuple(slice(g, n - g if g else None) for n in spatial)
    f = pdf[inner]
    c = torch.tensor(st.stencil_entries, dtype=torch.float64, device="cuda")[:, :D]
    want_rho = 1.0 + f.sum(-1)
    want_u = (f @ c + 0.5 * torch.tensor([1e-3, 2e-3, 0.0][:D], dtype=torch.float64, device="cuda")) / want_rho[..., None]
    # sums of 19 terms of 0.01 in FP64, then one rounding to the output type
    tol = 1e-15 * 32 if dtype == torch.float64 else 2.0 ** -24
    for got, want in ((rho, want_rho), (dev, want_rho - 1.0), (u, want_u)):
        assert float((got[inner].double() - want).abs().max()) <= tol * 1.5
        # nothing beside the interior is written
        outside = torch.ones(got.shape, dtype=torch.bool, device="cuda")
        outside[inner] = False
        assert bool((got[outside] == 7.0).all())


def test_other_outputs_take_the_staged_way():
    st = LBStencil("D3Q19")
    m = create_lb_method(LBMConfig(stencil=st, relaxation_rate=1.7))
    pdf = create_pdf_array((20, 9, 7), 19, 0, "float32")
    pdf.copy_(0.01 * torch.randn(pdf.shape, device="cuda"))
    get = compile_macroscopic_values_getter(m, ["density", "velocity"], ghost_layers=0)
    rho, u = torch.empty(20, 9, 7, device="cuda"), torch.empty(20, 9, 7, 3, device="cuda")
    get(pdf, density=rho, velocity=u)
    rho16, u16 = torch.empty_like(rho, dtype=torch.float16), torch.empty_like(u, dtype=torch.float64)
    get(pdf, density=rho16, velocity=u16)      # an FP16 field, and two types at once
    assert torch.equal(rho16, rho.half()) or float((rho16.float() - rho).abs().max()) <= 2.0 ** -11
    assert torch.equal(u16.float(), u)
