"""lbm355_boundary_groups: NoSlip and UBB groups that share launches leave what each group's own launch leaves."""
import ctypes

import pytest
import torch

from lbmpy_amd import LBStencil
from lbmpy_amd import _native as nat

pytestmark = pytest.mark.gpu

DTYPES = {torch.float64: nat.F64, torch.float32: nat.F32, torch.float16: nat.F16}
KINDS = [0, 1, 1, 0, 1, 0, 1]          # 0: NoSlip, 1: UBB
SIZES = {"D2Q9": (40, 17, 1), "D3Q19": (9, 12, 7), "D3Q27": (5, 4, 6)}


@pytest.mark.parametrize("stencil", list(SIZES))
@pytest.mark.parametrize("dtype", list(DTYPES), ids=str)
@pytest.mark.parametrize("pattern", range(10))
def test_groups_equal_single_launches(pattern, dtype, stencil):
    st = LBStencil(stencil)
    size, flat = SIZES[stencil], stencil == "D2Q9"
    gen = torch.Generator().manual_seed(pattern)
    full = [n + 2 for n in size[:2]] + [1 if flat else size[2] + 2]
    links = [(x, y, z, d) for x in range(1, size[0] + 1) for y in range(1, size[1] + 1)
             for z in ([0] if flat else range(1, size[2] + 1)) for d, c in enumerate(st.stencil_entries)
             if any(not 1 <= p + e <= n for p, e, n in zip((x, y, z), c, size))]
    order = torch.randperm(len(links), generator=gen)
    links = torch.tensor(links, dtype=torch.int32)[order]
    # group lengths: one link, blocks not quite, just and more than filled, none
    cuts = [1, 255, 0, 256, 257, 3] if len(links) > 800 else [1, 30, 0, 40, 25, 3]
    groups = list(torch.split(links, cuts + [len(links) - sum(cuts)]))
    groups = [g.contiguous().cuda() for g in groups]
    data = [None] * len(groups)
    data[4] = (0.05 * torch.randn((len(groups[4]), 3), generator=gen, dtype=torch.float64)).cuda()
    descs = (nat.BoundaryDesc * len(groups))()
    for k, d in enumerate(descs):
        d.stencil, d.pattern, d.store_dtype = nat.STENCIL_NAMES[stencil], pattern, DTYPES[dtype]
        d.kind = KINDS[k]
        d.nx, d.ny, d.nz = size
        d.ghost_layers = 1
        d.flags = nat.FLAG_ZERO_CENTERED | (nat.FLAG_COMPRESSIBLE if k == 6 else 0)
        d.stride_y, d.stride_z, d.stride_q = full[0], 0 if flat else full[0] * full[1], full[0] * full[1] * full[2]
        d.velocity[0], d.velocity[1] = 0.03 * k, -0.01
        d.density = 1.1 if k == 1 else 0.0
    state = (1e-2 * torch.randn((st.Q, full[2], full[1], full[0]), generator=gen)).to(dtype).cuda()
    lib, stream = nat.load(), nat.current_stream_handle()
    pointers = [(ctypes.c_void_p(g.data_ptr()), ctypes.c_void_p(v.data_ptr() if v is not None else None))
                for g, v in zip(groups, data)]
    want, got = state.clone(), state.clone()
    for k, (l, v) in enumerate(pointers):
        nat.check(lib.lbm355_boundary_links(ctypes.byref(descs[k]), ctypes.c_void_p(want.data_ptr()), l, len(groups[k]), v,
                                            stream))
    n = len(groups)
    nat.check(lib.lbm355_boundary_groups(descs, n, ctypes.c_void_p(got.data_ptr()),
                                         (ctypes.c_void_p * n)(*[l.value for l, _ in pointers]),
                                         (ctypes.c_int64 * n)(*[len(g) for g in groups]),
                                         (ctypes.c_void_p * n)(*[v.value for _, v in pointers]), stream))
    assert torch.equal(got, want) and not torch.equal(want, state)
    assert bool(torch.isfinite(want.float()).all())
