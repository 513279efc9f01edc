"""The sweeps choose how they number the cells and reach memory by the populations' size and alignment (sweep_launch in
csrc/sweep_cell.h).  Small domains, which the oracle pins, all take the same way; here large ones take each of the
others.  A state that repeats along the periodic axes must evolve exactly as one of its tiles."""
import numpy as np
import pytest
import torch

from lbmpy_amd import LBMConfig, LBStencil, CreateKernelConfig, Target, Timestep, Method, create_lb_function

pytestmark = pytest.mark.gpu

# (stencil, method, pattern, dtype, tile, repeats, ghost layers, walls in y)
CASES = [
    # rows on lines of their own, x-shifts through LDS
    ("D3Q27", Method.CUMULANT, "aa", "float32", (64, 16, 16), (2, 9, 9), 0, False),
    ("D3Q19", Method.TRT, "pull", "float64", (64, 16, 12), (3, 5, 6), 0, True),
    ("D3Q27", Method.CUMULANT, "esotwist", "float32", (64, 16, 16), (3, 8, 8), 0, False),
    # rows of whole wavefronts, too long for the row kernels, or FP16
    ("D3Q19", Method.TRT, "pull", "float32", (64, 8, 16), (9, 6, 6), 0, False),
    ("D3Q27", Method.CUMULANT, "esopull", "float32", (64, 8, 16), (9, 12, 6), 0, False),
    ("D3Q27", Method.CUMULANT, "aa", "float16", (64, 16, 16), (2, 9, 9), 0, False),
    # consecutive cells, rows of any length
    ("D3Q27", Method.CUMULANT, "aa", "float32", (25, 16, 16), (8, 8, 8), 0, False),
    ("D3Q19", Method.MRT, "pull", "float32", (25, 16, 16), (5, 2, 20), 0, True),
    ("D3Q19", Method.SRT, "pull", "float16", (41, 16, 16), (3, 6, 12), 0, False),
    # rows that share lines: ghost layers, or planes of odd size
    ("D3Q19", Method.TRT, "aa", "float64", (33, 15, 17), (4, 9, 9), 0, True),
    ("D3Q27", Method.CUMULANT, "pull", "float32", (64, 11, 13), (1, 10, 9), 1, False),
    ("D3Q19", Method.CENTRAL_MOMENT, "esopush", "float32", (37, 15, 21), (5, 9, 8), 0, False),
]


def _run(case, shape, storage, steps):
    stencil, method, pattern, dtype, _, _, g, walls = case
    kw = dict(stencil=LBStencil(stencil), method=method, relaxation_rate=1.7, streaming_pattern=pattern,
              compressible=method in (Method.CUMULANT, Method.CENTRAL_MOMENT))
    cfg = CreateKernelConfig(target=Target.GPU, data_type=dtype,
                             compute_type="float64" if dtype == "float64" else "float32", ghost_layers=g)
    times = (None,) if pattern in ("pull", "push") else (Timestep.ODD, Timestep.EVEN)
    ks = [create_lb_function(lbm_config=LBMConfig(**kw) if t is None else LBMConfig(**kw, timestep=t), config=cfg)
          for t in times]
    full = torch.zeros((storage.shape[0],) + tuple(n + 2 * g for n in shape[::-1]), dtype=storage.dtype, device="cuda")
    inner = (slice(None),) + (slice(g, -g if g else None),) * 3
    full[inner] = storage
    a, b = full, torch.zeros_like(full)
    for k in ks:
        k.set_faces(["periodic", "noslip" if walls else "periodic", "periodic"])
    for s in range(steps):
        if len(ks) == 1:
            ks[0](src=a.permute(3, 2, 1, 0), dst=b.permute(3, 2, 1, 0))
            a, b = b, a
        else:
            ks[s % 2](src=a.permute(3, 2, 1, 0))
    return a[inner]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:4]) + "-" + "x".join(map(str, c[4])))
def test_large_domain_equals_its_tile(case):
    tile, reps, walls = case[4], case[5], case[7]
    if walls:                      # the walls stand at the ends: the tile spans the whole axis
        tile, reps = (tile[0], tile[1] * reps[1], tile[2]), (reps[0], 1, reps[2])
    q = {"D3Q19": 19, "D3Q27": 27}[case[0]]
    rng = np.random.default_rng(7)
    state = torch.from_numpy(1e-3 * rng.standard_normal((q,) + tile[::-1])).to(getattr(torch, case[3])).cuda()
    shape = tuple(n * r for n, r in zip(tile, reps))
    # beyond what the sweeps take for fitting the Infinity Cache
    arrays = 2 if case[2] == "pull" else 1
    bound = (1 if arrays == 2 or case[3] == "float16" else 2) * (128 << 20)
    assert arrays * q * int(np.prod(shape)) * state.element_size() > bound
    want = _run(case, tile, state, 4)
    got = _run(case, shape, state.repeat(1, *reps[::-1]), 4)
    assert torch.equal(got, want.repeat(1, *reps[::-1]))
    assert not torch.equal(want, state) and bool(torch.isfinite(want.double()).all())
