"""Getter, conserved sums and the non-finite count on fields with long axes, and of 2^31 cells and more, which kernels that
number their cells in 32 bits take in boxes.  Reference: the few populations that are not 0, by hand."""
import numpy as np
import pytest
import torch

from lbmpy_amd import CreateKernelConfig, LBMConfig, LBStencil, Target, compile_macroscopic_values_getter, \
    compile_macroscopic_values_setter, create_lb_function, create_lb_method
from lbmpy_amd.sweep import create_pdf_array

pytestmark = pytest.mark.gpu


def _objects(stencil, dtype):
    cfg = LBMConfig(stencil=LBStencil(stencil), relaxation_rate=1.7, compressible=True)
    kernel = create_lb_function(lbm_config=cfg, config=CreateKernelConfig(
        target=Target.GPU, data_type=dtype, compute_type="float64" if dtype == "float64" else "float32", ghost_layers=0))
    return create_lb_method(cfg), kernel


@pytest.mark.parametrize("order", ["f", "c"])
@pytest.mark.parametrize("shape", [(4, 70000), (70000, 4), (3, 70000, 2), (2, 3, 70000)])
def test_long_axes(shape, order):
    D = len(shape)
    m, kernel = _objects("D2Q9" if D == 2 else "D3Q19", "float64")
    rng = np.random.default_rng(3)
    rho = torch.from_numpy(1 + 0.01 * rng.standard_normal(shape)).cuda()
    u = torch.from_numpy(0.02 * rng.standard_normal(shape + (D,))).cuda()
    pdf = create_pdf_array(shape, m.stencil.Q, 0, "float64")
    compile_macroscopic_values_setter(m, {"density": rho, "velocity": u}, ghost_layers=0)(pdf)

    def out(*n):
        return torch.zeros(n, dtype=torch.float64, device="cuda") if order == "c" else \
            torch.zeros(n[::-1], dtype=torch.float64, device="cuda").permute(*reversed(range(len(n))))
    got_rho, got_u = out(*shape), out(*shape, D)
    compile_macroscopic_values_getter(m, ["density", "velocity"], ghost_layers=0)(pdf, density=got_rho, velocity=got_u)
    # an FP64 equilibrium and its moments: 19 terms of at most 1/3, each way
    assert float((got_rho - rho).abs().max()) <= 1e-14 and float((got_u - u).abs().max()) <= 1e-14
    assert abs(kernel.conserved(pdf)[0] - float(rho.sum())) <= 1e-12 * rho.numel()
    assert kernel.nonfinite_count(pdf) == 0


@pytest.mark.parametrize("stencil,shape", [("D2Q9", (46400, 46400)), ("D3Q19", (1300, 1290, 1290))])
def test_more_than_2_31_cells(stencil, shape):
    D = len(shape)
    cells = int(np.prod(shape, dtype=np.int64))
    assert cells > 2 ** 31
    m, kernel = _objects(stencil, "float16")
    q = m.stencil.Q
    need = (2 * q + 4) * cells
    if torch.cuda.mem_get_info()[0] + torch.cuda.memory_reserved() < need + (4 << 30):
        pytest.skip("not enough GPU memory")
    pdf = create_pdf_array(shape, q, 0, "float16")
    rows = (2 ** 31 - 1) // shape[0]            # cells on both sides of a box's end, and the ends of the field
    at = [(0,) * D, tuple(n - 1 for n in shape), (5, rows - 1) if D == 2 else (5, 7, rows // shape[1] - 1),
          (5, rows) if D == 2 else (5, 7, rows // shape[1])]
    for k, cell in enumerate(at):
        pdf[cell + (1 + k,)] = 0.25 * (k + 1)
    c = np.array(m.stencil.stencil_entries)
    sums = kernel.conserved(pdf)
    assert sums[0] == cells + 2.5
    np.testing.assert_array_equal(sums[1:1 + D], sum(0.25 * (k + 1) * c[1 + k][:D] for k in range(4)))
    rho = torch.zeros(shape[::-1], dtype=torch.float32, device="cuda").permute(*reversed(range(D)))
    compile_macroscopic_values_getter(m, ["density_deviation"], ghost_layers=0)(pdf, density_deviation=rho)
    assert [float(rho[cell]) for cell in at] == [0.25, 0.5, 0.75, 1.0]
    storage = rho.permute(*reversed(range(D)))
    assert sum(int(torch.count_nonzero(s)) for s in storage.split(256)) == 4
    del rho, storage
    for k, cell in enumerate(at):
        pdf[cell + (k,)] = float("nan") if k % 2 else float("inf")
    assert kernel.nonfinite_count(pdf) == 4
    del pdf
    torch.cuda.empty_cache()
