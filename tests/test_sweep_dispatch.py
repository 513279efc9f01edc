"""The access mode that lbm355_sweep chooses (choose_access in csrc/sweep_cell.h), by size, alignment, pattern and walls.
Host code only: the arrays are addresses that nothing reads."""
import ctypes
import os

import numpy as np
import pytest

from lbmpy_amd import _native as nat

ROWS, WAVES, LINES, CACHED, SHARED = nat.ACCESS_ROWS, nat.ACCESS_WAVES, nat.ACCESS_LINES, nat.ACCESS_CACHED, \
    nat.ACCESS_SHARED
STENCILS = {"D2Q9": (nat.D2Q9, 9), "D3Q19": (nat.D3Q19, 19), "D3Q27": (nat.D3Q27, 27)}
PATTERNS = {"pull": nat.PULL, "push": nat.PUSH, "even": nat.AA_EVEN, "odd": nat.AA_ODD, "esotwist": nat.INPLACE_EVEN["esotwist"],
            "esopull": nat.INPLACE_EVEN["esopull"]}
TYPES = {"f64": nat.F64, "f32": nat.F32, "f16": nat.F16}


@pytest.fixture(scope="module")
def lib():
    from lbmpy_amd.csrc.build import library_path
    if not os.path.exists(library_path()):
        pytest.skip("liblbm355.so not built (run __graft_entry__.build())")
    return nat.load()


def _mode(lib, stencil, pattern, dtype, shape, g=0, walls=False, pad=0, shift=0, closure=False, cumulant=False):
    d = nat.SweepDesc()
    d.stencil, q = STENCILS[stencil]
    d.family = nat.FAMILY_CUMULANT if closure or cumulant else nat.FAMILY_MOMENT
    d.pattern, d.store_dtype = PATTERNS[pattern], TYPES[dtype]
    d.compute_dtype = nat.F64 if dtype == "f64" else nat.F32
    shape = tuple(shape) + (1,) * (3 - len(shape))
    D = 2 if stencil == "D2Q9" else 3
    d.nx, d.ny, d.nz = shape
    d.ghost_layers = g
    for a in range(3):
        d.face[a] = nat.FACE_GHOST if g and a < D else nat.FACE_NOSLIP if walls and a == 1 else nat.FACE_PERIODIC
    d.stride_y = shape[0] + 2 * g + pad
    d.stride_z = d.stride_y * (shape[1] + 2 * g)
    d.stride_q = d.stride_z * (shape[2] + 2 * g) if D == 3 else d.stride_z
    d.tables = 4096
    if closure:
        d.flags = nat.FLAG_LEARNED_CLOSURE
        d.closure = 4096
    src = (1 << 40) + shift
    dst = src if pattern not in ("pull", "push") else (1 << 41) + shift
    return lib.lbm355_sweep_access(ctypes.byref(d), src, dst)


@pytest.mark.parametrize("args,want", [
    # what the caches hold: 128 MiB for two arrays and FP16, 256 MiB in place
    (("D3Q27", "odd", "f32", (128, 128, 128)), CACHED), (("D3Q27", "even", "f64", (64, 64, 64)), CACHED),
    (("D3Q19", "pull", "f32", (64, 64, 64)), CACHED), (("D3Q27", "even", "f16", (128, 128, 128)), CACHED),
    (("D2Q9", "pull", "f64", (900, 900)), CACHED), (("D3Q19", "pull", "f32", (128, 128, 96)), ROWS),
    # in place up to 768 MiB without walls: regular accesses, although the lines would allow streaming
    (("D3Q27", "odd", "f32", (128, 144, 144)), SHARED), (("D3Q27", "even", "f32", (200, 128, 128)), SHARED),
    (("D3Q27", "esotwist", "f32", (192, 128, 128)), SHARED), (("D3Q27", "esopull", "f32", (576, 96, 96)), SHARED),
    (("D3Q27", "odd", "f64", (128, 128, 128)), SHARED), (("D2Q9", "even", "f64", (2048, 2048)), SHARED),
    # beyond: rows, wavefronts, consecutive cells
    (("D3Q27", "odd", "f32", (256, 192, 160)), ROWS), (("D3Q27", "even", "f32", (256, 192, 160)), WAVES),
    (("D3Q27", "even", "f32", (200, 224, 224)), LINES), (("D3Q27", "odd", "f32", (200, 224, 224)), SHARED),
    (("D3Q27", "esotwist", "f32", (192, 256, 224)), ROWS), (("D3Q27", "esopull", "f32", (576, 144, 128)), WAVES),
    (("D3Q27", "esopull", "f32", (200, 224, 224)), SHARED), (("D3Q27", "push", "f32", (256, 192, 160)), ROWS),
    # FP16 has no row kernels for pull and AA; a block a row in AA odd
    (("D3Q27", "odd", "f16", (256, 256, 256)), WAVES), (("D3Q19", "odd", "f16", (512, 256, 256)), SHARED),
    (("D3Q19", "odd", "f16", (250, 200, 180)), SHARED), (("D3Q27", "even", "f16", (256, 256, 256)), WAVES),
    (("D3Q19", "pull", "f16", (123, 96, 192)), LINES), (("D3Q27", "esotwist", "f16", (256, 256, 256)), ROWS),
    # two dimensions
    (("D2Q9", "pull", "f64", (512, 4096)), ROWS), (("D2Q9", "pull", "f64", (1024, 1024)), WAVES),
    (("D2Q9", "pull", "f64", (1000, 1024)), LINES), (("D2Q9", "pull", "f64", (1000, 1001)), SHARED),
    # in place up to 576 MiB
    (("D2Q9", "even", "f32", (4000, 4000)), SHARED), (("D2Q9", "even", "f32", (4096, 4096)), WAVES),
    (("D2Q9", "odd", "f64", (512, 14000)), SHARED), (("D2Q9", "odd", "f64", (512, 16400)), ROWS),
    (("D2Q9", "esopull", "f32", (4096, 4096)), SHARED), (("D2Q9", "odd", "f64", (448, 32768)), ROWS), (("D2Q9", "even", "f32", (4096, 8192)), WAVES),
])
def test_chosen_mode(lib, args, want):
    assert _mode(lib, *args) == want


def test_alignment_walls_and_padding(lib):
    big = ("D3Q27", "even", "f32", (256, 192, 160))
    assert _mode(lib, *big, shift=64) == SHARED and _mode(lib, *big, shift=128) == WAVES
    assert _mode(lib, "D3Q27", "even", "f32", (256, 192, 160), g=1) == SHARED
    # rows on lines of their own: 30 elements of padding beside two ghost cells, and the first cell on a line
    padded = dict(g=1, pad=30)
    first = 4 * (1 + 288 + 288 * 194)
    assert _mode(lib, *big, **padded) == SHARED and _mode(lib, *big, **padded, shift=-first % 128) == WAVES
    # walls: streamed from 256 MiB on
    assert _mode(lib, "D3Q19", "odd", "f32", (192, 160, 192), walls=True) == ROWS
    assert _mode(lib, "D3Q19", "odd", "f32", (192, 160, 192)) == SHARED
    # the learned closure needs whole wavefronts in every mode
    for n, pattern, want in ((128, "odd", CACHED), (192, "even", SHARED), (256, "even", WAVES), (256, "odd", ROWS)):
        assert _mode(lib, "D3Q27", pattern, "f32", (n, n, n), closure=True) == want
    assert _mode(lib, "D3Q27", "even", "f32", (200, 128, 128), closure=True) < 0
    for kw in (dict(cumulant=True), dict(walls=True)):
        assert _mode(lib, "D3Q27", "odd", "f16", (256, 256, 256), **kw) == SHARED


def test_cases_of_the_large_domain_tests(lib):
    """Which modes the large domains of the other tests take."""
    from tests import test_gpu_sweep_access as access, test_gpu_sweep_turns as turns
    got = set()
    for stencil, method, pattern, dtype, tile, reps, g, walls in access.CASES + turns.CASES:
        shape = tuple(int(n) for n in np.multiply(tile, reps))
        for p in ("odd", "even") if pattern == "aa" else (pattern,):
            if p in PATTERNS:
                got.add((p, _mode(lib, stencil, p, {"float64": "f64", "float32": "f32", "float16": "f16"}[dtype], shape,
                                  g=0, walls=walls)))
    assert {("odd", ROWS), ("even", WAVES), ("even", LINES), ("odd", SHARED), ("even", SHARED), ("pull", ROWS),
            ("pull", WAVES), ("pull", LINES), ("pull", SHARED), ("esotwist", ROWS), ("esopull", WAVES)} <= got
