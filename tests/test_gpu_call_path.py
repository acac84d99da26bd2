"""The C++ call path between the Python classes and the C ABI: what it refuses, and what
becomes of a result's buffers."""

from __future__ import annotations

import gc

import pytest
import torch

import nacho_amd as na

pytestmark = pytest.mark.gpu

I, F = torch.int32, torch.float32


def _operands(kind, gpu, n):
    """Two equal operands with n entries, all in row (or slice) 0."""
    crd = torch.arange(n, dtype=I, device=gpu)
    zero = torch.zeros(n, dtype=I, device=gpu)
    pos = torch.tensor([0, n], dtype=I, device=gpu)
    one = torch.zeros(1, dtype=I, device=gpu)
    unit = torch.tensor([0, 1], dtype=I, device=gpu)
    val = torch.arange(n, dtype=F, device=gpu) + 1

    def make():
        if kind == "csr":
            return na.CSR_gpu(pos.clone(), crd.clone(), val.clone(), [1, n + 1])
        if kind == "coo":
            return na.COO_gpu(zero.clone(), crd.clone(), val.clone(), [1, n + 1])
        if kind == "coo3":
            return na.COO3_gpu(zero.clone(), zero.clone(), crd.clone(), val.clone(), [1, 1, n + 1])
        if kind == "dcsr":
            return na.DCSR_gpu(one.clone(), pos.clone(), crd.clone(), val.clone(), [1, n + 1])
        return na.CSF3_gpu(one.clone(), unit.clone(), one.clone(), pos.clone(), crd.clone(),
                           val.clone(), [1, 1, n + 1])

    return make(), make()


ADD = {"csr": "gpu_csr_add_f32", "coo": "gpu_coo_add_f32", "coo3": "gpu_coo3d_add_f32",
       "dcsr": "gpu_dcsr_add_f32", "csf3": "gpu_csf_add_f32"}


@pytest.mark.parametrize("kind", sorted(ADD))
def test_each_class_through_the_call_path(kind, gpu):
    a, b = _operands(kind, gpu, 1000)
    z = getattr(na, ADD[kind])(a, b)
    assert type(z) is type(a) and z.device == a.device
    for name, dtype in a._fields:
        buf = getattr(z, name)
        assert buf.dtype == dtype and buf.device == gpu and buf.is_contiguous()
        expect = getattr(a, name) * (2 if name == "values" else 1)
        assert torch.equal(buf, expect)
    assert z.shape.tolist() == a.shape.tolist()


@pytest.mark.parametrize("kind", sorted(ADD))
def test_operand_whose_buffers_disagree_is_refused(kind, gpu):
    for name in [n for n, _ in _operands(kind, gpu, 4)[0]._fields]:
        a, b = _operands(kind, gpu, 64)
        buf = getattr(b, name)
        buf.resize_(buf.numel() - 1)  # a buffer changed in place after the checks on creation
        with pytest.raises(ValueError):
            getattr(na, ADD[kind])(a, b)


def test_wrong_class_is_refused(gpu):
    a, _ = _operands("csr", gpu, 8)
    b, _ = _operands("coo", gpu, 8)
    with pytest.raises(TypeError, match="operand b must be CSR_gpu, got COO_gpu"):
        na.gpu_csr_add_f32(a, b)


def test_empty_result_has_empty_buffers(gpu):
    a, _ = _operands("csr", gpu, 16)
    b = na.CSR_gpu(torch.tensor([0, 0], dtype=I, device=gpu), torch.empty(0, dtype=I, device=gpu),
                   torch.empty(0, dtype=F, device=gpu), [1, 17])
    z = na.gpu_csr_mul_f32(a, b)
    assert z.dim_j_offsets.tolist() == [0, 0]
    for buf, dtype in ((z.dim_j_indices, I), (z.values, F)):
        assert buf.numel() == 0 and buf.dtype == dtype and buf.device == gpu


def test_buffer_returns_to_the_allocator_with_its_last_view(gpu):
    a, b = _operands("csr", gpu, 1 << 20)
    na.gpu_csr_add_f32(a, b)
    gc.collect()
    torch.cuda.synchronize()
    idle = na.cached_bytes()
    z = na.gpu_csr_add_f32(a, b)
    view = z.values[5:9]
    expect = view.tolist()
    del z
    held = idle - na.cached_bytes()
    assert held >= (1 << 20) * 4, "the values' buffer went back while a view of it lived"
    na.gpu_csr_add_f32(b, a)
    assert view.tolist() == expect
    del view
    assert na.cached_bytes() >= idle


def test_exception_of_an_entry_point(gpu, tmp_path):
    """A C++ exception out of the library (no host memory, say) arrives as a Python one, and the
    interpreter goes on."""
    import ctypes
    import subprocess

    from nacho_amd import _lib, ops

    src = tmp_path / "throws.cpp"
    src.write_text('#include <new>\nextern "C" int throws() { throw std::bad_alloc(); }\n')
    lib = tmp_path / "throws.so"
    subprocess.run(["g++", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    address = ctypes.cast(ctypes.CDLL(str(lib)).throws, ctypes.c_void_p).value
    a, b = _operands("csr", gpu, 8)
    bridge = _lib.load_bridge()
    args = [x for t in (a, b) for x in (ops._CSR.kind, ops._CSR.buffers(t), t._dims)]
    for _ in range(3):
        with pytest.raises(RuntimeError, match="bad_alloc"):
            bridge.invoke(address, ops._CSR.kind, 256, 256, 0, 0, *args)
    assert na.gpu_csr_add_f32(a, b).values.tolist() == (2 * a.values).tolist()
