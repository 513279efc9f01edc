"""Every access mode of the sweeps (lbm355_sweep_with_access), at sizes where lbm355_sweep itself would take only the
cached one: each family, pattern and type in every mode its kernels come in, against the cached mode; and the oracle
tests of small domains once more in the streamed modes."""
import contextlib
import functools
import itertools

import numpy as np
import pytest
import torch

from lbmpy_amd import CreateKernelConfig, LBMConfig, LBStencil, Method, SubgridScaleModel, Target, Timestep, \
    create_lb_function
from lbmpy_amd import _native as nat

pytestmark = pytest.mark.gpu

MODES = {"rows": nat.ACCESS_ROWS, "waves": nat.ACCESS_WAVES, "lines": nat.ACCESS_LINES, "cached": nat.ACCESS_CACHED,
         "shared": nat.ACCESS_SHARED}


class _Forced:
    """The library with lbm355_sweep in one mode, where the sweep has it; `taken` lists the modes that ran."""

    def __init__(self, lib, access):
        self._lib, self._access, self.taken = lib, access, []

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def lbm355_sweep(self, d, src, dst, rho, u, stream):
        rc = self._lib.lbm355_sweep_with_access(d, src, dst, rho, u, self._access, stream)
        if rc == 2 and b"access mode" in self._lib.lbm355_last_error():       # LBM355_ERR_UNSUPPORTED
            self.taken.append(self._lib.lbm355_sweep_access(d, src, dst))
            return self._lib.lbm355_sweep(d, src, dst, rho, u, stream)
        self.taken.append(self._access)
        return rc


@contextlib.contextmanager
def forced(monkeypatch, mode):
    lib = _Forced(nat.load(), MODES[mode])
    with monkeypatch.context() as m:
        m.setattr(nat, "load", lambda *a: lib)
        yield lib


RATES27 = [0.0, 0, 0, 0, 1.7, 1.6, 1.5, 1.4, 1.3, 1.2, 1.1, 1.0, 0.9, 0.8, 0.7, 0.6, 0.5, 0.4, 0.3, 0.35, 0.45, 0.55,
           0.65, 0.75, 0.85, 0.95, 1.05]
CUMULANT = dict(method=Method.CUMULANT, compressible=True)
FAMILIES = {
    "D2Q9-trt": ("D2Q9", dict(method=Method.TRT, relaxation_rates=[1.8, 1.1], force=(1e-4, 0))),
    "D2Q9-central": ("D2Q9", dict(method=Method.CENTRAL_MOMENT, relaxation_rate=1.7, compressible=True)),
    "D3Q19-mrt": ("D3Q19", dict(method=Method.MRT, relaxation_rate=1.8, force=(1e-5, 0, 0))),
    "D3Q19-central": ("D3Q19", dict(method=Method.CENTRAL_MOMENT, relaxation_rate=1.7, compressible=True)),
    "D3Q27-srt": ("D3Q27", dict(method=Method.SRT, relaxation_rate=1.6)),
    "D3Q27-central": ("D3Q27", dict(method=Method.CENTRAL_MOMENT, relaxation_rate=1.7, compressible=True)),
    "cumulant": ("D3Q27", dict(CUMULANT, relaxation_rate=1.9, force=(1e-5, 2e-5, 0))),
    "cumulant-rates": ("D3Q27", dict(CUMULANT, relaxation_rates=RATES27)),
    "cumulant-smagorinsky": ("D3Q27", dict(CUMULANT, relaxation_rate=1.9,
                                           subgrid_scale_model=(SubgridScaleModel.SMAGORINSKY, 0.16))),
    "cumulant-corrected": ("D3Q27", dict(CUMULANT, relaxation_rate=1.9, galilean_correction=True,
                                         fourth_order_correction=0.01)),
    "cumulant-monomial": ("D3Q27", dict(method=Method.MONOMIAL_CUMULANT, relaxation_rate=1.6, compressible=True)),
    "closure": ("D3Q27", dict(CUMULANT, relaxation_rate=1.9)),
}
EPS = {"float64": 2.0 ** -52, "float32": 2.0 ** -23, "float16": 2.0 ** -23}


@functools.lru_cache(maxsize=None)
def _closure():
    from lbmpy_amd.closure import ClosureModel
    return ClosureModel(seed=4, nu_scale=1e-3)


@functools.lru_cache(maxsize=None)
def _kernels(family, pattern, dtype, g):
    stencil, kw = FAMILIES[family]
    cfg = CreateKernelConfig(target=Target.GPU, data_type=dtype,
                             compute_type="float64" if dtype == "float64" else "float32", ghost_layers=g)
    times = [{}] if pattern in ("pull", "push") else [{"timestep": Timestep.ODD}, {"timestep": Timestep.EVEN}]
    ks = [create_lb_function(lbm_config=LBMConfig(stencil=LBStencil(stencil), streaming_pattern=pattern, **kw, **t),
                             config=cfg) for t in times]
    if family == "closure":
        for k in ks:
            k.set_closure(_closure())
    return ks


def _run(family, pattern, dtype, g, walls, state, steps=4):
    ks = _kernels(family, pattern, dtype, g)
    D = state.dim() - 1
    for k in ks:
        k.set_faces(["periodic", "noslip" if walls else "periodic"] + ["periodic"] * (D - 2))
    full = torch.zeros((state.shape[0],) + tuple(n + 2 * g for n in state.shape[1:]), dtype=state.dtype, device="cuda")
    inner = (slice(None),) + (slice(g, -g if g else None),) * D
    full[inner] = state
    order = tuple(range(D, -1, -1))
    a, b = full.permute(order), torch.zeros_like(full).permute(order)
    for s in range(steps):
        if len(ks) == 1:
            ks[0](src=a, dst=b)
            a, b = b, a
        else:
            ks[s % 2](src=a)
    return a.permute(order)[inner]


def _compare(monkeypatch, family, pattern, dtype, g, walls, shape):
    q = {"D2Q9": 9, "D3Q19": 19, "D3Q27": 27}[FAMILIES[family][0]]
    rng = np.random.default_rng(7)
    state = torch.from_numpy(1e-2 * rng.standard_normal((q,) + shape[::-1])).to(getattr(torch, dtype)).cuda()
    with forced(monkeypatch, "cached") as lib:
        want = _run(family, pattern, dtype, g, walls, state).double()
    assert set(lib.taken) == {nat.ACCESS_CACHED} and bool(torch.isfinite(want).all())
    assert float((want - state.double()).abs().max()) > 1e-3
    # the modes share their arithmetic up to the contraction of products and sums: some hundred roundings a step of
    # numbers of the state's size; stored in FP16, one that lands on the other side of a rounding boundary
    tol = 256 * EPS[dtype] * float(want.abs().max())
    if dtype == "float16":
        tol += 2.0 ** -9 * float(want.abs().max())
    ran = set()
    for mode in ("rows", "waves", "lines", "shared"):
        with forced(monkeypatch, mode) as lib:
            got = _run(family, pattern, dtype, g, walls, state).double()
        ran.update(lib.taken)
        assert float((got - want).abs().max()) <= tol, mode
    return ran


def _patterns(family):
    return ("pull", "aa") if family == "closure" else ("pull", "aa", "push", "esotwist", "esopull", "esopush")


@pytest.mark.parametrize("dtype", ["float64", "float32", "float16"])
@pytest.mark.parametrize("family,pattern", [(f, p) for f in FAMILIES for p in _patterns(f)])
def test_modes_agree(monkeypatch, family, pattern, dtype):
    if family == "closure" and dtype != "float32":
        pytest.skip("the learned closure runs in FP32")
    shape = (64, 6) if family.startswith("D2Q9") else (64, 5, 3)
    for g, walls in [(0, False), (1, False)] + [(0, True)] * (pattern in ("pull", "aa")):
        ran = _compare(monkeypatch, family, pattern, dtype, g, walls, shape)
        want = {nat.ACCESS_SHARED, nat.ACCESS_WAVES}
        if pattern in ("pull", "aa"):
            want.add(nat.ACCESS_LINES)
        if dtype != "float16" or pattern not in ("pull", "aa"):
            want.add(nat.ACCESS_ROWS)
        assert want <= ran


# rows of two blocks, rows too long for the row kernels, rows of no whole wavefront, one cell
@pytest.mark.parametrize("shape", [(320, 3, 2), (512, 2, 2), (576, 2, 2), (35, 5, 4), (65, 1, 3), (1, 1, 1)])
@pytest.mark.parametrize("family,pattern,dtype", [("cumulant", "aa", "float32"), ("cumulant", "pull", "float16"),
                                                  ("D3Q19-mrt", "pull", "float64"), ("D3Q19-mrt", "esopull", "float32"),
                                                  ("D2Q9-trt", "pull", "float64"), ("D2Q9-trt", "aa", "float32")])
def test_modes_agree_for_other_rows(monkeypatch, family, pattern, dtype, shape):
    ran = _compare(monkeypatch, family, pattern, dtype, 0, False, shape[:2] if family.startswith("D2Q9") else shape)
    assert (nat.ACCESS_WAVES in ran) == (shape[0] % 64 == 0)
    assert nat.ACCESS_ROWS not in ran or shape[0] % 64 == 0 and shape[0] <= 512


def _calls(test):
    """The keyword arguments that a test's parametrize marks give it."""
    sets = []
    for mark in (m for m in getattr(test, "pytestmark", []) if m.name == "parametrize"):
        names = [n.strip() for n in mark.args[0].split(",")]
        sets.append([dict(zip(names, v if len(names) > 1 else (v,))) for v in mark.args[1]])
    return [{k: v for part in combo for k, v in part.items()} for combo in itertools.product(*sets)]


ORACLE_TESTS = [("test_gpu_parity", "test_row_lds_kernels_fp64", "rows"),
                ("test_gpu_parity", "test_row_lds_kernels_fp64", "waves"),
                ("test_gpu_parity", "test_moment_family_fp64", "lines"),
                ("test_gpu_parity", "test_central_moment_family_fp64", "lines"),
                ("test_gpu_parity", "test_cumulant_smagorinsky_fp64", "lines"),
                ("test_gpu_parity", "test_moment_family_fp64", "shared"),
                ("test_gpu_streaming_patterns", "test_pattern_row_staged_sweep_fp64_matches_oracle", "rows"),
                ("test_gpu_streaming_patterns", "test_pattern_row_staged_sweep_fp64_matches_oracle", "waves"),
                ("test_gpu_streaming_patterns", "test_pattern_sweep_fp64_matches_oracle", "shared"),
                ("test_gpu_cumulant_corrections", "test_corrected_cumulant_fp64_matches_oracle", "lines"),
                ("test_gpu_cumulant_corrections", "test_corrected_cumulant_fp32_close_to_fp64", "rows"),
                ("test_gpu_cumulant_sets", "test_monomial_cumulant_fp64", "lines"),
                ("test_gpu_closure", "test_fused_sweep_matches_oracle_collision", "rows"),
                ("test_gpu_closure", "test_fused_sweep_matches_oracle_collision", "waves"),
                ("test_gpu_closure", "test_fused_sweep_matches_oracle_collision", "shared")]


@pytest.mark.parametrize("module,name,mode", ORACLE_TESTS)
def test_oracle_in_mode(monkeypatch, module, name, mode):
    test = getattr(__import__("tests." + module, fromlist=[name]), name)
    with forced(monkeypatch, mode) as lib:
        for kwargs in _calls(test):
            test(**kwargs)
    assert MODES[mode] in lib.taken


def test_refusals():
    k = _kernels("cumulant", "aa", "float32", 0)[1]
    pdf = torch.zeros(27, 3, 5, 35, device="cuda").permute(3, 2, 1, 0)
    k.set_faces(["periodic"] * 3)
    d = k.descriptor(pdf, {})
    lib = nat.load()
    run = (lambda access: lib.lbm355_sweep_with_access(d, pdf.data_ptr(), pdf.data_ptr(), None, None, access, None))
    assert run(nat.ACCESS_ROWS) == run(nat.ACCESS_WAVES) == 2 and run(-1) == 1 and run(5) == 2
    assert float(pdf.abs().max()) == 0.0


@pytest.mark.parametrize("pattern,mode", [("pull", "rows"), ("push", "rows"), ("esopull", "rows"), ("pull", "waves")])
def test_padded_rows_on_lines(pattern, mode):
    """Rows with ghost layers and padding, whose cells start on lines, are streamed; without padding they are not."""
    family, dtype = ("cumulant", "float32") if mode == "rows" else ("D3Q19-mrt", "float16")
    nx, ny, nz, q = (128, 120, 100, 27) if mode == "rows" else (128, 160, 160, 19)
    if pattern == "esopull":
        nx, ny, nz = 256, 192, 160
    ks = _kernels(family, pattern, dtype, 1)
    for k in ks:
        k.set_faces(["periodic"] * 3)
    per_line = 128 // torch.empty(0, dtype=getattr(torch, dtype)).element_size()
    full = (nx + 2, ny + 2, nz + 2)

    def arrays(padded):
        sy = -(-full[0] // per_line) * per_line if padded else full[0]
        sz = sy * full[1]
        sq = sz * full[2]
        first = -(1 + sy + sz) % per_line if padded else 0
        out = []
        for _ in range(2 if pattern in ("pull", "push") else 1):
            flat = torch.zeros(q * sq + first, dtype=getattr(torch, dtype), device="cuda")
            out.append(flat.as_strided(full + (q,), (1, sy, sz, sq), first))
        return out

    g = torch.Generator(device="cuda").manual_seed(5)
    state = 1e-2 * torch.randn((nx, ny, nz, q), generator=g, device="cuda")
    results = []
    for padded in (True, False):
        a = arrays(padded)
        a[0][1:-1, 1:-1, 1:-1] = state.to(a[0].dtype)
        chosen = set()
        for s in range(2):
            k = ks[s % len(ks)]
            chosen.add(nat.load().lbm355_sweep_access(k.descriptor(a[0], {}), a[0].data_ptr(), a[-1].data_ptr()))
            if len(a) == 2:
                k(src=a[0], dst=a[1])
                a = a[::-1]
            else:
                k(src=a[0])
        assert chosen == ({MODES[mode]} if padded else {nat.ACCESS_SHARED})
        results.append(a[0][1:-1, 1:-1, 1:-1].double())
    tol = 128 * EPS[dtype] * float(results[1].abs().max()) + (2.0 ** -10 * float(results[1].abs().max())
                                                              if dtype == "float16" else 0.0)
    assert float((results[0] - results[1]).abs().max()) <= tol and float((results[1] - state).abs().max()) > 1e-3
