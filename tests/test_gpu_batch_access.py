"""A batch reaches memory by its size and its members' alignment: in the caches, past them, or with lines that wavefronts
share (batch_access in csrc/batch.hip).  In each, every member must end as its own kernel alone leaves it."""
import pytest
import torch

from lbmpy_amd import LBMConfig, LBStencil, CreateKernelConfig, Target, Timestep, Method, create_lb_function
from lbmpy_amd.batch import BatchedSweep
from lbmpy_amd.sweep import create_pdf_array

pytestmark = pytest.mark.gpu

MIXES = {"cached": [(17, 9, 5), (64, 8, 8), (1, 3, 2)],
         "shared": [(130, 101, 190), (97, 188, 110), (33, 5, 5), (150, 190, 77)],
         "lines": [(128, 96, 64), (64, 64, 64), (128, 128, 192), (192, 128, 128)]}
LAUNCHES = [(256, 0, 0), (128, 3, 1), (64, 0, 1), (192, 1, 0)]


@pytest.mark.parametrize("launch", LAUNCHES)
@pytest.mark.parametrize("mix", list(MIXES))
@pytest.mark.parametrize("dtype", ["float32", "float64", "float16"])
@pytest.mark.parametrize("pattern", ["pull", "aa"])
def test_members_equal_single_sweeps(pattern, dtype, mix, launch):
    cfg = CreateKernelConfig(target=Target.GPU, data_type=dtype,
                             compute_type="float64" if dtype == "float64" else "float32", ghost_layers=0)
    g = torch.Generator(device="cuda").manual_seed(3)
    members = []
    for k, shape in enumerate(MIXES[mix]):
        kw = dict(stencil=LBStencil("D3Q19"), method=Method.TRT, relaxation_rate=1.5 + 0.1 * k, streaming_pattern=pattern)
        times = [{}] if pattern == "pull" else [{"timestep": Timestep.ODD}, {"timestep": Timestep.EVEN}]
        kernels = [create_lb_function(lbm_config=LBMConfig(**kw, **t), config=cfg) for t in times]
        for kern in kernels:
            kern.set_faces(["periodic", "noslip", "periodic"])
        a = create_pdf_array(shape, 19, 0, dtype)
        a.copy_(1e-2 * torch.randn(a.shape, generator=g, device="cuda", dtype=torch.float32))
        b = torch.zeros_like(a) if pattern == "pull" else a
        members.append((kernels, a, b, a.clone(), torch.zeros_like(a)))
    batch = BatchedSweep([m[0][-1] for m in members], [m[1] for m in members],
                         [m[2] for m in members] if pattern == "pull" else None)
    batch.launch = launch
    batch.run(3)
    for k, ((kernels, _, _, p, q), got) in enumerate(zip(members, batch.current_arrays())):
        for t in range(3):
            if pattern == "pull":
                kernels[0](src=p, dst=q)
                p, q = q, p
            else:
                kernels[t % 2](src=p)
        assert torch.equal(got, p), k
