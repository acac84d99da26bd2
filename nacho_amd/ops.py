"""`gpu_<kernel>_f32` entry points with the reference's Python signatures.

The reference's generated wrapper (src/backend/generate_bindings.cpp:288-327) unwraps each
operand class into the kernel's tensor struct, calls `<k>::<k>_gpu_i32_f32(operands...,
num_blocks, threads_per_block)` and adopts the returned buffers.  These functions do the
same through the C ABI of libnacho_hip.so: borrow operand buffers, call the entry point on
torch's current stream, adopt the result buffers.  Those steps are C++ (bridge/bridge.cpp);
what an operand may be is checked there, and named here when it is refused.  There is no CPU
fallback: a missing library raises.
"""

from __future__ import annotations

import ctypes
import operator

import torch

from . import _device, _lib
from .tensors import COO3_gpu, COO_gpu, CSF3_gpu, CSR64_gpu, CSR_gpu, DCSR_gpu, Scalar_gpu


def _p(t: torch.Tensor):
    return ctypes.c_void_p(_device.ptr(t))


def _same_device(*tensors):
    device = tensors[0].device
    for t in tensors[1:]:
        if t.device != device:
            raise ValueError(f"operands on different devices: {device} and {t.device}")
    return device


# ---- operand checks ------------------------------------------------------------------

def _buffers(t):
    return [getattr(t, name) for name in t._attributes]


def _check_csr(t: CSR_gpu) -> None:
    rows = t._dims[0]
    if t.dim_j_offsets.numel() != rows + 1:
        raise ValueError(f"CSR_gpu: dim_j_offsets has {t.dim_j_offsets.numel()} entries, "
                         f"expected rows + 1 = {rows + 1}")
    if t.values.numel() != t.dim_j_indices.numel():
        raise ValueError("CSR_gpu: dim_j_indices and values differ in length")


def _check_coo(t) -> None:
    if any(x.numel() != t.values.numel() for x in _buffers(t)):
        raise ValueError(f"{type(t).__name__}: coordinate and value arrays differ in length")


def _check_dcsr(t: DCSR_gpu) -> None:
    ni = t.dim_i_indices.numel()
    if t.dim_j_offsets.numel() != ni + 1:
        raise ValueError(f"DCSR_gpu: dim_j_offsets has {t.dim_j_offsets.numel()} entries, "
                         f"expected stored rows + 1 = {ni + 1}")
    if t.values.numel() != t.dim_j_indices.numel():
        raise ValueError("DCSR_gpu: dim_j_indices and values differ in length")


def _check_csf3(t: CSF3_gpu) -> None:
    ni, nj = t.dim_i_indices.numel(), t.dim_j_indices.numel()
    if t.dim_j_offsets.numel() != ni + 1 or t.dim_k_offsets.numel() != nj + 1:
        raise ValueError("CSF3_gpu: offsets arrays must have parent length + 1 entries")
    if t.values.numel() != t.dim_k_indices.numel():
        raise ValueError("CSF3_gpu: dim_k_indices and values differ in length")


class _Operand:
    """How the call path takes a class: its number there (enum Kind in bridge/bridge.cpp), its
    buffers as a tuple, and the check that names what is wrong with a refused one."""

    __slots__ = ("cls", "kind", "buffers", "check")

    def __init__(self, cls, kind, check=None):
        self.cls, self.kind, self.check = cls, kind, check
        self.buffers = operator.attrgetter(*cls._attributes)


_CSR, _COO = _Operand(CSR_gpu, 0, _check_csr), _Operand(COO_gpu, 1, _check_coo)
_COO3, _DCSR = _Operand(COO3_gpu, 2, _check_coo), _Operand(DCSR_gpu, 3, _check_dcsr)
_CSF3 = _Operand(CSF3_gpu, 4, _check_csf3)
_CSR64, _SCALAR = _Operand(CSR64_gpu, 5), _Operand(Scalar_gpu, 6)  # results only


# ---- input validation ----------------------------------------------------------------

_VALIDATE = False


def set_validation(enable: bool) -> None:
    """Validation mode: when enabled, every `gpu_` entry point first checks its CSR operands
    on the device (nacho_validate_csr) and raises ValueError for a malformed one.  Off by
    default: like the reference's generated code, the kernels trust operand contents."""
    global _VALIDATE
    _VALIDATE = bool(enable)


def validate_csr(t: CSR_gpu) -> None:
    """Check a CSR operand against the input contract (pos[0] == 0, pos non-decreasing,
    pos[rows] == nnz, 0 <= crd < columns, crd strictly increasing per row); raises
    ValueError if it is malformed."""
    if not isinstance(t, CSR_gpu):
        raise TypeError(f"validate_csr: expected CSR_gpu, got {type(t).__name__}")
    _check_csr(t)
    n = t.values.numel()
    desc = _lib.CsrDesc(*t._dims, _p(t.dim_j_offsets), n, _p(t.dim_j_indices), _p(t.values), n)
    with _device.on_device(t.device):
        rc = _lib.load().nacho_validate_csr(ctypes.byref(desc),
                                            ctypes.c_void_p(_device.current_stream(t.device)))
    if rc == -4:  # NACHO_ERR_MALFORMED_INPUT
        raise ValueError("CSR operand violates the input contract (offsets, column range or "
                         "per-row order)")
    _lib.check(rc, "nacho_validate_csr")


def _validate_all(*operands):
    for t in operands:
        if isinstance(t, CSR_gpu):
            validate_csr(t)


# ---- generic call --------------------------------------------------------------------

_ENTRIES: dict = {}
_bridge = None


def _entry(name) -> int:
    """Address of the library's entry point `name` (looked up once)."""
    global _bridge
    address = _ENTRIES.get(name)
    if address is None:
        lib = _lib.load()
        if _bridge is None:
            _bridge = _lib.load_bridge()
        fn = getattr(lib, name, None)
        if fn is None:
            raise RuntimeError(f"{name} is not exported by {_lib.LIBRARY_PATH.name}")
        address = _ENTRIES[name] = ctypes.cast(fn, ctypes.c_void_p).value
    return address


def _refuse(entry, operands, kinds):
    """Raise for operands that the call path did not take, naming what is wrong."""
    for t, kind in zip(operands, kinds):
        kind.check(t)
    _same_device(*(buf for t, kind in zip(operands, kinds) for buf in kind.buffers(t)))
    raise ValueError(f"{entry}: an operand has more than 2^31 - 1 entries")


def _call(entry, operands, kinds, result, num_blocks, threads_per_block):
    """One entry point on `operands` (of `kinds`, in order), giving a `result`."""
    args = []
    for t, kind in zip(operands, kinds):
        if not isinstance(t, kind.cls):
            raise TypeError(f"{entry}: operand {'abc'[len(args) // 3]} must be "
                            f"{kind.cls.__name__}, got {type(t).__name__}")
        args += (kind.kind, kind.buffers(t), t._dims)
    if _VALIDATE:
        _validate_all(*operands)
    device = _same_device(*operands)
    address = _entry(entry)
    with _device.on_device(device):
        stream = _device.current_stream(device)
        z = _bridge.invoke(address, result.kind, int(num_blocks), int(threads_per_block), stream,
                           device.index, *args)
        if type(z) is tuple:
            return result.cls._trusted(z[0], z[1], device)
        if z is None:
            _refuse(entry, operands, kinds)
        _lib.check(z, entry)


def gpu_csr_add_f32(a: CSR_gpu, b: CSR_gpu, num_blocks: int = 256,
                    threads_per_block: int = 256) -> CSR_gpu:
    """Z = a + b (sorted union per row; explicit zeros kept).  compiler.cpp:112."""
    return _call("nacho_gpu_csr_add_f32", (a, b), (_CSR, _CSR), _CSR, num_blocks, threads_per_block)


def gpu_csr_add_3_f32(a: CSR_gpu, b: CSR_gpu, c: CSR_gpu, num_blocks: int = 256,
                      threads_per_block: int = 256) -> CSR_gpu:
    """Z = a + b + c (sorted union of three; values (a + b) + c over the present operands).
    compiler.cpp:114."""
    return _call("nacho_gpu_csr_add_3_f32", (a, b, c), (_CSR, _CSR, _CSR), _CSR, num_blocks,
                 threads_per_block)


def gpu_sssmm_f32(a: CSR_gpu, b: CSR_gpu, c: CSR_gpu, num_blocks: int = 256,
                  threads_per_block: int = 256) -> CSR_gpu:
    """Masked SpGEMM Z_ik = sum_j a_ij b_jk c_ik over the entries of c that a product reaches.
    compiler.cpp:150-153."""
    return _call("nacho_gpu_sssmm_f32", (a, b, c), (_CSR, _CSR, _CSR), _CSR, num_blocks,
                 threads_per_block)


def gpu_csr_mul_f32(a: CSR_gpu, b: CSR_gpu, num_blocks: int = 256,
                    threads_per_block: int = 256) -> CSR_gpu:
    """Z = a * b elementwise (sorted intersection per row).  compiler.cpp:116."""
    return _call("nacho_gpu_csr_mul_f32", (a, b), (_CSR, _CSR), _CSR, num_blocks, threads_per_block)


def gpu_coo_add_f32(a: COO_gpu, b: COO_gpu, num_blocks: int = 256,
                    threads_per_block: int = 256) -> COO_gpu:
    """Z = a + b over COO (union of (i, j)).  compiler.cpp:118."""
    return _call("nacho_gpu_coo_add_f32", (a, b), (_COO, _COO), _COO, num_blocks, threads_per_block)


def gpu_coo_mul_f32(a: COO_gpu, b: COO_gpu, num_blocks: int = 256,
                    threads_per_block: int = 256) -> COO_gpu:
    """Z = a * b over COO (intersection of (i, j)).  compiler.cpp:120."""
    return _call("nacho_gpu_coo_mul_f32", (a, b), (_COO, _COO), _COO, num_blocks, threads_per_block)


def gpu_coo3d_add_f32(a: COO3_gpu, b: COO3_gpu, num_blocks: int = 256,
                      threads_per_block: int = 256) -> COO3_gpu:
    """Z = a + b over COO3 (union of (i, j, k)).  compiler.cpp:138."""
    return _call("nacho_gpu_coo3d_add_f32", (a, b), (_COO3, _COO3), _COO3, num_blocks,
                 threads_per_block)


def gpu_dcsr_add_f32(a: DCSR_gpu, b: DCSR_gpu, num_blocks: int = 256,
                     threads_per_block: int = 256) -> DCSR_gpu:
    """Z = a + b over DCSR (union of row ids, then of each row's columns).
    compiler.cpp:124."""
    return _call("nacho_gpu_dcsr_add_f32", (a, b), (_DCSR, _DCSR), _DCSR, num_blocks,
                 threads_per_block)


def gpu_dcsr_mul_f32(a: DCSR_gpu, b: DCSR_gpu, num_blocks: int = 256,
                     threads_per_block: int = 256) -> DCSR_gpu:
    """Z = a * b over DCSR: rows stored in both operands, each with the intersection of its
    columns (kept when that is empty).  compiler.cpp:126."""
    return _call("nacho_gpu_dcsr_mul_f32", (a, b), (_DCSR, _DCSR), _DCSR, num_blocks,
                 threads_per_block)


def gpu_dcsr_mul_without_recursive_partitioning_f32(
        a: DCSR_gpu, b: DCSR_gpu, num_blocks: int = 256,
        threads_per_block: int = 256) -> DCSR_gpu:
    """The same product as gpu_dcsr_mul_f32 (the reference variant differs only in how it
    partitions work).  compiler.cpp:128-133."""
    return _call("nacho_gpu_dcsr_mul_without_recursive_partitioning_f32", (a, b),
                 (_DCSR, _DCSR), _DCSR, num_blocks, threads_per_block)


def gpu_csf_add_f32(a: CSF3_gpu, b: CSF3_gpu, num_blocks: int = 256,
                    threads_per_block: int = 256) -> CSF3_gpu:
    """Z = a + b over CSF3 (union at every level).  compiler.cpp:135."""
    return _call("nacho_gpu_csf_add_f32", (a, b), (_CSF3, _CSF3), _CSF3, num_blocks,
                 threads_per_block)


def gpu_coo_csr_add_f32(a: CSR_gpu, b: COO_gpu, num_blocks: int = 256,
                        threads_per_block: int = 256) -> CSR_gpu:
    """Z = a + b for a CSR a and a COO b (sorted, no duplicates), giving CSR.
    compiler.cpp:122."""
    return _call("nacho_gpu_coo_csr_add_f32", (a, b), (_CSR, _COO), _CSR, num_blocks,
                 threads_per_block)


def gpu_inner_prod_f32(a: CSF3_gpu, b: CSF3_gpu, num_blocks: int = 256,
                       threads_per_block: int = 256) -> Scalar_gpu:
    """z = sum_ijk a_ijk * b_ijk over CSF3 operands (float32 products summed in float64,
    rounded once).  compiler.cpp:141."""
    return _call("nacho_gpu_inner_prod_f32", (a, b), (_CSF3, _CSF3), _SCALAR, num_blocks,
                 threads_per_block)


def gpu_inner_prod_coo_f32(a: COO3_gpu, b: COO3_gpu, num_blocks: int = 256,
                           threads_per_block: int = 256) -> Scalar_gpu:
    """The same inner product over COO3 operands.  compiler.cpp:143."""
    return _call("nacho_gpu_inner_prod_coo_f32", (a, b), (_COO3, _COO3), _SCALAR, num_blocks,
                 threads_per_block)


def gpu_spgemm_f32(a: CSR_gpu, b: CSR_gpu, num_blocks: int = 256,
                   threads_per_block: int = 256) -> CSR_gpu:
    """Z_ik = sum_j a_ij b_jk (ESC SpGEMM), int32 result.  compiler.cpp:145-148."""
    return _call("nacho_gpu_spgemm_f32", (a, b), (_CSR, _CSR), _CSR, num_blocks, threads_per_block)


def gpu_spgemm64_f32(a: CSR_gpu, b: CSR_gpu, num_blocks: int = 256,
                     threads_per_block: int = 256) -> CSR64_gpu:
    """The same product with int64 result offsets, for results beyond 2^31 entries."""
    return _call("nacho_gpu_spgemm64_f32", (a, b), (_CSR, _CSR), _CSR64, num_blocks,
                 threads_per_block)


def release_cached_memory() -> None:
    """Return the default allocator's cached, unused device buffers to the driver."""
    _lib.check(_lib.load().nacho_release_cached_memory(), "nacho_release_cached_memory")


def set_cache_limit(nbytes: int | None) -> None:
    """Cap the bytes the library's caching allocator keeps for reuse (None: no cap, the
    default).  Past the cap, released buffers go back to the driver (after a device
    synchronise), so that torch's allocator in the same process can use that memory."""
    limit = ctypes.c_size_t(-1).value if nbytes is None else int(nbytes)
    if limit < 0:
        raise ValueError("cache limit must be >= 0")
    _lib.check(_lib.load().nacho_set_cache_limit(limit), "nacho_set_cache_limit")


def cached_bytes() -> int:
    """Bytes the library's caching allocator holds for reuse now."""
    return int(_lib.load().nacho_cached_bytes())


def set_kernel_timing(enable: bool) -> None:
    _lib.load().nacho_set_kernel_timing(1 if enable else 0)


def last_kernel_ms() -> float:
    return float(_lib.load().nacho_last_kernel_ms())
