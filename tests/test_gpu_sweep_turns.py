"""Sweeps of populations that exceed the Infinity Cache: up to 768 MiB in place they use the caches, every other sweep
backwards; beyond, or with walls, they stream past them; of arrays whose lines wavefronts share, two beyond 1 GiB keep one
direction (meets_cached and cached_anyway in csrc/sweep_cell.h).  A state that repeats along the periodic axes must evolve
exactly as one of its tiles."""
import numpy as np
import pytest
import torch

from lbmpy_amd import Method
from tests.test_gpu_sweep_access import _run

pytestmark = pytest.mark.gpu

# (stencil, method, pattern, dtype, tile, repeats, ghost layers, walls in y)
CASES = [
    # in place, backwards: the last block partly filled, and filled; both sides of 768 MiB
    ("D3Q27", Method.CUMULANT, "aa", "float32", (25, 15, 17), (7, 10, 9), 0, False),
    ("D3Q27", Method.CUMULANT, "aa", "float64", (64, 16, 16), (2, 8, 8), 0, False),
    ("D3Q19", Method.TRT, "esotwist", "float32", (40, 16, 16), (6, 13, 13), 0, False),
    ("D3Q27", Method.CUMULANT, "aa", "float32", (64, 16, 16), (4, 12, 10), 0, False),
    ("D3Q27", Method.CUMULANT, "aa", "float32", (64, 16, 16), (4, 12, 11), 0, False),
    # streamed
    ("D3Q27", Method.CUMULANT, "aa", "float32", (25, 16, 16), (8, 14, 14), 0, False),
    ("D3Q27", Method.CUMULANT, "esotwist", "float32", (64, 16, 16), (3, 16, 14), 0, False),
    ("D3Q27", Method.CUMULANT, "esopull", "float32", (64, 8, 16), (9, 18, 8), 0, False),
    ("D3Q19", Method.TRT, "aa", "float32", (64, 16, 12), (3, 10, 16), 0, True),
    # two arrays, on both sides of 1 GiB
    ("D3Q19", Method.TRT, "pull", "float32", (33, 15, 17), (8, 10, 9), 1, True),
    ("D3Q19", Method.TRT, "pull", "float32", (33, 15, 17), (8, 10, 12), 1, False),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:4]) + "-" + "x".join(map(str, c[4] + c[5])))
def test_large_domain_equals_its_tile(case):
    tile, reps, walls = case[4], case[5], case[7]
    if walls:                      # the walls stand at the ends: the tile spans the whole axis
        tile, reps = (tile[0], tile[1] * reps[1], tile[2]), (reps[0], 1, reps[2])
    q = {"D3Q19": 19, "D3Q27": 27}[case[0]]
    rng = np.random.default_rng(7)
    state = torch.from_numpy(1e-3 * rng.standard_normal((q,) + tile[::-1])).to(getattr(torch, case[3])).cuda()
    shape = tuple(n * r for n, r in zip(tile, reps))
    want = _run(case, tile, state, 4)
    got = _run(case, shape, state.repeat(1, *reps[::-1]), 4)
    assert torch.equal(got, want.repeat(1, *reps[::-1]))
    assert not torch.equal(want, state) and bool(torch.isfinite(want.double()).all())
