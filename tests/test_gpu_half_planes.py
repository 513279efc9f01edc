"""FP16 population planes of an odd number of elements, and arrays that start on an odd element: half of their planes
do not start on a dword.  Every cell must evolve exactly as in an array whose planes all do."""
import pytest
import torch

from lbmpy_amd import LBMConfig, LBStencil, CreateKernelConfig, Target, Timestep, Method, create_lb_function

pytestmark = pytest.mark.gpu


def _planes(shape, q, gap, start):
    """[q, z, y, x] view: planes `gap` elements longer than their cells, the first at element `start`."""
    n = shape[0] * shape[1] * shape[2] + gap
    storage = torch.full((start + q * n,), 7.0, dtype=torch.float16, device="cuda")
    view = storage.as_strided((q, shape[2], shape[1], shape[0]), (n, shape[0] * shape[1], shape[0], 1), start)
    return storage, view


def _run(pattern, walls, state, shape, gap, start):
    cfg = CreateKernelConfig(target=Target.GPU, data_type="float16", compute_type="float32", ghost_layers=0)
    kw = dict(stencil=LBStencil("D3Q19"), method=Method.TRT, relaxation_rate=1.7, streaming_pattern=pattern)
    times = ({},) if pattern == "pull" else ({"timestep": Timestep.ODD}, {"timestep": Timestep.EVEN})
    ks = [create_lb_function(lbm_config=LBMConfig(**kw, **t), config=cfg) for t in times]
    for k in ks:
        k.set_faces(["periodic", "noslip" if walls else "periodic", "periodic"])
    (sa, a), (sb, b) = (_planes(shape, 19, gap, start) for _ in range(2))
    a.copy_(state)
    for s in range(4):
        if pattern == "pull":
            ks[0](src=a.permute(3, 2, 1, 0), dst=b.permute(3, 2, 1, 0))
            a, b, sa, sb = b, a, sb, sa
        else:
            ks[s % 2](src=a.permute(3, 2, 1, 0))
    return a.clone(), sa


@pytest.mark.parametrize("shape", [(16, 9, 4), (17, 9, 5), (33, 5, 5), (1, 3, 1), (65, 3, 7)])
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("pattern", ["pull", "aa"])
def test_odd_planes_equal_even_ones(pattern, walls, shape):
    g = torch.Generator(device="cuda").manual_seed(11)
    state = (1e-2 * torch.randn((19,) + shape[::-1], generator=g, device="cuda")).half()
    n = shape[0] * shape[1] * shape[2]
    want, _ = _run(pattern, walls, state, shape, n % 2, 0)
    for gap, start in ((0, 0), (1 - n % 2, 1)):
        got, storage = _run(pattern, walls, state, shape, gap, start)
        assert torch.equal(got, want), (gap, start)
        outside = torch.cat([storage[:start]] + [storage[start + i * (n + gap) + n:start + (i + 1) * (n + gap)] for i in range(19)])
        assert bool((outside == 7.0).all())
