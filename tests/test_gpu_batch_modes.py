"""Batches beyond the caches (batch_access in csrc/batch.hip), for the families whose small batches take the cached way:
every member must end as its own kernel alone leaves it, one thread per cell (the row kernels may contract a sum otherwise:
D3Q27 FP64 with a rate per cumulant differs by an ulp in 3 of 1000 cells)."""
import numpy as np
import pytest
import torch

from lbmpy_amd import CreateKernelConfig, LBMConfig, LBStencil, Method, Target, Timestep, create_lb_function
from lbmpy_amd import _native as nat
from lbmpy_amd.batch import BatchedSweep
from lbmpy_amd.sweep import create_pdf_array

pytestmark = pytest.mark.gpu

RATES27 = [0.0, 0, 0, 0, 1.7, 1.6, 1.5, 1.4, 1.3, 1.2, 1.1, 1.0, 0.9, 0.8, 0.7, 0.6, 0.5, 0.4, 0.3, 0.35, 0.45, 0.55,
           0.65, 0.75, 0.85, 0.95, 1.05]
FAMILIES = {
    "D2Q9-srt": ("D2Q9", dict(method=Method.SRT, relaxation_rate=1.6)),
    "D2Q9-central": ("D2Q9", dict(method=Method.CENTRAL_MOMENT, relaxation_rate=1.7, compressible=True)),
    "D3Q19-central": ("D3Q19", dict(method=Method.CENTRAL_MOMENT, relaxation_rate=1.7, compressible=True)),
    "D3Q27-srt": ("D3Q27", dict(method=Method.SRT, relaxation_rate=1.6)),
    "cumulant": ("D3Q27", dict(method=Method.CUMULANT, compressible=True, relaxation_rate=1.9)),
    "cumulant-rates": ("D3Q27", dict(method=Method.CUMULANT, compressible=True, relaxation_rates=RATES27)),
}
# members whose cells start on lines, and members whose rows share lines
SHAPES = {(2, True): [(1024, 1024), (576, 900), (1024, 1280)], (2, False): [(1001, 1023), (577, 801), (3, 5), (1025, 1300)],
          (3, True): [(128, 96, 64), (64, 64, 128), (192, 64, 64)], (3, False): [(101, 97, 90), (63, 60, 61), (3, 1, 2), (150, 61, 77)]}
HALF_CACHE = 128 << 20


def _sweep(kernel, src, dst):
    d = kernel.descriptor(src, {})
    nat.check(nat.load().lbm355_sweep_with_access(d, src.data_ptr(), dst.data_ptr(), None, None, nat.ACCESS_CACHED,
                                                  nat.current_stream_handle()))


@pytest.mark.parametrize("lines", [True, False], ids=["lines", "shared"])
@pytest.mark.parametrize("dtype", ["float64", "float32", "float16"])
@pytest.mark.parametrize("pattern", ["pull", "aa"])
@pytest.mark.parametrize("family", list(FAMILIES))
def test_members_equal_single_sweeps(family, pattern, dtype, lines):
    stencil, kw = FAMILIES[family]
    D, q = {"D2Q9": (2, 9), "D3Q19": (3, 19), "D3Q27": (3, 27)}[stencil]
    cfg = CreateKernelConfig(target=Target.GPU, data_type=dtype,
                             compute_type="float64" if dtype == "float64" else "float32", ghost_layers=0)
    times = [{}] if pattern == "pull" else [{"timestep": Timestep.ODD}, {"timestep": Timestep.EVEN}]
    kernels = [create_lb_function(lbm_config=LBMConfig(stencil=LBStencil(stencil), streaming_pattern=pattern, **kw, **t),
                                  config=cfg) for t in times]
    for k in kernels:
        k.set_faces(["periodic", "noslip"] + ["periodic"] * (D - 2))
    shapes = list(SHAPES[D, lines])
    per_cell = (2 if pattern == "pull" else 1) * q * torch.empty(0, dtype=getattr(torch, dtype)).element_size()
    while per_cell * sum(int(np.prod(s)) for s in shapes) <= HALF_CACHE:
        shapes.append(shapes[len(shapes) % 3])
    g = torch.Generator(device="cuda").manual_seed(3)
    members = []
    for shape in shapes:
        a = create_pdf_array(shape, q, 0, dtype)
        a.copy_(1e-2 * torch.randn(a.shape, generator=g, device="cuda", dtype=torch.float32))
        members.append((a, torch.zeros_like(a) if pattern == "pull" else a, a.clone(), torch.zeros_like(a)))
    batch = BatchedSweep([kernels[-1]] * len(members), [m[0] for m in members],
                         [m[1] for m in members] if pattern == "pull" else None)
    batch.run(3)
    for k, ((_, _, p, o), got) in enumerate(zip(members, batch.current_arrays())):
        for t in range(3):
            if pattern == "pull":
                _sweep(kernels[0], p, o)
                p, o = o, p
            else:
                _sweep(kernels[t % 2], p, p)
        assert bool(torch.isfinite(got.double()).all()) and torch.equal(got, p), k


def test_two_arrays_beyond_turns():
    """Two arrays of more than 1 GiB keep one direction."""
    cfg = CreateKernelConfig(target=Target.GPU, data_type="float32", ghost_layers=0)
    k = create_lb_function(lbm_config=LBMConfig(stencil=LBStencil("D3Q27"), streaming_pattern="pull",
                                                **FAMILIES["cumulant"][1]), config=cfg)
    k.set_faces(["periodic"] * 3)
    g = torch.Generator(device="cuda").manual_seed(4)
    members = []
    for shape in [(150, 120, 110), (151, 121, 111), (149, 119, 109)]:
        a = create_pdf_array(shape, 27, 0, "float32")
        a.copy_(1e-2 * torch.randn(a.shape, generator=g, device="cuda"))
        members.append((a, torch.zeros_like(a), a.clone(), torch.zeros_like(a)))
    assert 2 * sum(m[0].numel() * 4 for m in members) > (1 << 30)
    batch = BatchedSweep([k] * 3, [m[0] for m in members], [m[1] for m in members])
    batch.run(3)
    for (_, _, p, o), got in zip(members, batch.current_arrays()):
        for _ in range(3):
            _sweep(k, p, o)
            p, o = o, p
        assert torch.equal(got, p)
