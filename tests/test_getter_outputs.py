"""The macroscopic getter writes its outputs directly only where every element written is its own."""
import ctypes
import os

import pytest
import torch

from lbmpy_amd import _native as nat

SHAPE = (6, 5, 4)


@pytest.fixture(scope="module", autouse=True)
def _library():
    from lbmpy_amd.csrc.build import library_path
    if not os.path.exists(library_path()):
        pytest.skip("liblbm355.so not built (run __graft_entry__.build())")


def _own_memory(pdfs, scalars, velocity):
    """lbm355_fields_apart for these tensors (host code, which reads no element)."""
    D = pdfs.dim() - 1
    d, o = nat.SweepDesc(), nat.MacroscopicOut()
    d.stencil = nat.D2Q9 if D == 2 else nat.D3Q19
    d.store_dtype = o.dtype = nat.F32
    d.nx, d.ny, d.nz = tuple(pdfs.shape[:D]) + (1,) * (3 - D)
    d.stride_y, d.stride_z, d.stride_q = pdfs.stride(1), pdfs.stride(2) if D == 3 else 0, pdfs.stride(D)
    for name, t in zip(("density", "density_deviation"), scalars):
        setattr(o, name, t.data_ptr())
        assert t.stride() == scalars[0].stride()
        for a in range(D):
            o.scalar_stride[a] = t.stride(a)
    if velocity is not None:
        o.velocity = velocity.data_ptr()
        for a in range(D):
            o.vector_stride[a] = velocity.stride(a)
        o.vector_stride[3] = velocity.stride(D)
    return bool(nat.load().lbm355_fields_apart(ctypes.byref(d), pdfs.data_ptr(), ctypes.byref(o)))


def _pdfs(q=19, extra=0):
    return torch.zeros((q + extra,) + SHAPE[::-1]).permute(3, 2, 1, 0)


def _c(*shape):
    return torch.zeros(shape)


def _f(*shape):
    return torch.zeros(shape[::-1]).permute(*reversed(range(len(shape))))


def test_separate_fields():
    for make in (_c, _f):
        assert _own_memory(_pdfs(), [make(*SHAPE), make(*SHAPE)], make(*SHAPE, 3))
        assert _own_memory(_pdfs(), [], make(*SHAPE, 3)) and _own_memory(_pdfs(), [make(*SHAPE)], None)
    one = torch.zeros(1, 1, 1)
    assert _own_memory(torch.zeros(1, 1, 1, 19), [one], None)


def test_interleaved_components_are_separate():
    cell = _c(*SHAPE, 4)                       # [x, y, z][rho, u]
    assert _own_memory(_pdfs(), [cell[..., 0]], cell[..., 1:])
    assert _own_memory(_pdfs(), [cell[..., 3]], cell[..., :3])
    plane = _f(*SHAPE, 5)                      # one x-fastest plane per component
    assert _own_memory(_pdfs(), [plane[..., 0], plane[..., 4]], plane[..., 1:4])
    flat = torch.zeros(9, 7, 6).permute(2, 1, 0)
    cell = _c(6, 7, 3)
    assert _own_memory(flat, [cell[..., 0]], cell[..., 1:]) and _own_memory(flat, [_f(6, 7)], _c(6, 7, 2))
    assert not _own_memory(flat, [cell[..., 1]], cell[..., 1:])
    padded = torch.zeros(SHAPE[0] + 2, SHAPE[1], SHAPE[2] + 3)
    assert _own_memory(_pdfs(), [padded[1:-1, :, :SHAPE[2]]], None)


@pytest.mark.parametrize("extra", [0, 4])
def test_the_populations_own_memory_is_shared(extra):
    pdfs = _pdfs(extra=extra)
    f = pdfs[..., :19]
    assert not _own_memory(f, [f[..., 0]], None)
    assert not _own_memory(f, [], f[..., 5:8])
    assert not _own_memory(f, [_c(*SHAPE)], f[..., 16:19])
    if extra:
        assert _own_memory(f, [pdfs[..., 19]], pdfs[..., 20:23])


def test_shared_outputs():
    rho, u = _c(*SHAPE), _c(*SHAPE, 3)
    assert not _own_memory(_pdfs(), [rho, rho], u)
    assert not _own_memory(_pdfs(), [u[..., 1]], u)
    assert not _own_memory(_pdfs(), [_c(1, *SHAPE[1:]).expand(*SHAPE)], None)
    base = torch.zeros(200)
    sliding = base.as_strided(SHAPE, (1, 2, 3))   # elements of one field on top of each other
    assert not _own_memory(_pdfs(), [sliding], None)
    assert not _own_memory(_pdfs(), [], base.as_strided(SHAPE + (3,), (1, 6, 30, 6)))


@pytest.mark.gpu
def test_shared_memory_is_staged():
    from lbmpy_amd import LBMConfig, LBStencil, create_lb_method, compile_macroscopic_values_getter
    from lbmpy_amd.sweep import create_pdf_array
    m = create_lb_method(LBMConfig(stencil=LBStencil("D3Q19"), relaxation_rate=1.7, compressible=True))
    shape = (70, 33, 20)
    pdf = create_pdf_array(shape, 19, 0, "float32")
    pdf.copy_(0.01 * torch.randn(pdf.shape, device="cuda"))
    get = compile_macroscopic_values_getter(m, ["density", "density_deviation", "velocity"], ghost_layers=0)
    rho, dev = torch.empty(shape, device="cuda"), torch.empty(shape, device="cuda")
    u = torch.empty(shape + (3,), device="cuda")
    get(pdf, density=rho, density_deviation=dev, velocity=u)
    # into the populations themselves, and into one field after the other: the last one written stays
    own = pdf.clone(memory_format=torch.preserve_format)
    get(own, density=own[..., 0], density_deviation=own[..., 9], velocity=own[..., 1:4])
    assert torch.equal(own[..., 0], rho) and torch.equal(own[..., 9], dev) and torch.equal(own[..., 1:4], u)
    assert torch.equal(own[..., 10:], pdf[..., 10:])
    v = torch.empty(shape + (3,), device="cuda")
    get(pdf, density=v[..., 0], density_deviation=v[..., 0], velocity=v)
    assert torch.equal(v, u)
    # interleaved components take the direct way, and give the same
    cell = torch.empty(shape + (5,), device="cuda")
    get(pdf, density=cell[..., 0], density_deviation=cell[..., 4], velocity=cell[..., 1:4])
    assert torch.equal(cell[..., 0], rho) and torch.equal(cell[..., 4], dev) and torch.equal(cell[..., 1:4], u)


@pytest.mark.gpu
def test_torch_knows_of_the_write():
    from lbmpy_amd import LBMConfig, LBStencil, create_lb_method, compile_macroscopic_values_getter
    from lbmpy_amd.sweep import create_pdf_array
    m = create_lb_method(LBMConfig(stencil=LBStencil("D2Q9"), relaxation_rate=1.7))
    pdf = create_pdf_array((8, 7), 9, 0, "float64")
    pdf.fill_(0.01)
    get = compile_macroscopic_values_getter(m, ["density"], ghost_layers=0)
    rho = torch.ones(8, 7, dtype=torch.float64, device="cuda")
    w = torch.ones_like(rho, requires_grad=True)
    loss = (w * rho).sum()          # saves rho
    get(pdf, density=rho)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()
    # views with a pending negation, and tensors made in inference mode
    neg = torch.view_as_complex(torch.zeros(8, 7, 2, dtype=torch.float64, device="cuda")).conj().imag
    assert neg.is_neg()
    get(pdf, density=neg)
    assert torch.equal(neg, rho)
    with torch.inference_mode():
        frozen = torch.ones(8, 7, dtype=torch.float64, device="cuda")
        get(pdf, density=frozen)
    assert torch.equal(frozen, rho)
    with pytest.raises(RuntimeError):
        get(pdf, density=frozen)
