"""A call that fails half-way leaves nothing to the next one: a caller's allocator returns NULL at
each of the call's requests in turn, behind work that keeps the stream busy, and the same thread
then makes a correct call whose counts differ."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.helpers import csr_from_rows, random_csr
from tests.test_gpu_dcsr import run as run_dcsr
from tests.test_gpu_dcsr import want as want_dcsr
from tests.test_gpu_spgemm import run_and_check
from tests.test_gpu_sssmm import check as check_sssmm
from tests.test_gpu_sssmm import run as run_sssmm
from tests.test_oracle_dcsr import assert_dcsr_equal, random_dcsr

pytestmark = pytest.mark.gpu


class _FailingAllocator:
    """Device buffers from torch until request `fail_at` (never, if 0), NULL from then on."""

    def __init__(self, gpu, fail_at):
        from nacho_amd import _lib

        self.requests, self.keep, self.held = 0, [], set()

        def allocate(ctx, nbytes, stream):
            self.requests += 1
            if self.requests == fail_at:
                return None
            t = torch.empty(int(nbytes), dtype=torch.uint8, device=gpu)
            self.keep.append(t)  # (kept: what is queued may still use a released buffer)
            self.held.add(t.data_ptr())
            return t.data_ptr()

        def release(ctx, ptr, stream):
            self.held.remove(ptr)

        fields = dict(_lib.Allocator._fields_)
        self.struct = _lib.Allocator(None, fields["allocate"](allocate),
                                     fields["release"](release))


def _call(gpu, entry, descs, result, fail_at):
    from nacho_amd import _lib

    alloc = _FailingAllocator(gpu, fail_at)
    z = result()
    stream = torch.cuda.current_stream(gpu).cuda_stream
    rc = getattr(_lib.load(), entry)(*(ctypes.byref(d) for d in descs), ctypes.byref(z), 256, 256,
                                     ctypes.c_void_p(stream), ctypes.byref(alloc.struct))
    return rc, alloc, z


def _dev(gpu, keep, x):
    t = torch.from_numpy(np.ascontiguousarray(x)).to(gpu)
    keep.append(t)
    return t.data_ptr() if t.numel() else None


def _csr(gpu, keep, t, rows, cols):
    from nacho_amd import _lib

    pos, crd, val = t
    return _lib.CsrDesc(rows, cols, _dev(gpu, keep, pos), len(crd), _dev(gpu, keep, crd),
                        _dev(gpu, keep, val), len(val))


def _product_operands():
    """A large product with long rows, whose counts are all larger than the next call's."""
    rng = np.random.default_rng(2)
    n = 1500
    rows_a = [sorted({r, (r * 7 + 1) % n}) for r in range(n)]
    rows_a[100] = list(range(0, n, 2))
    a = csr_from_rows(n, n, rows_a)
    return n, a, random_csr(rng, n, 40000, 9 / 40000)


def _sssmm(gpu):
    from nacho_amd import _lib

    n, a, b = _product_operands()
    c = random_csr(np.random.default_rng(3), n, 40000, 20 / 40000)
    keep = []
    descs = (_csr(gpu, keep, a, n, n), _csr(gpu, keep, b, n, 40000), _csr(gpu, keep, c, n, 40000))
    return "nacho_gpu_sssmm_f32", descs, _lib.CsrDesc, keep


def _spgemm(gpu):
    from nacho_amd import _lib

    n, a, b = _product_operands()
    keep = []
    return ("nacho_gpu_spgemm_f32", (_csr(gpu, keep, a, n, n), _csr(gpu, keep, b, n, 40000)),
            _lib.CsrDesc, keep)


def _dcsr_mul(gpu):
    from nacho_amd import _lib

    rng = np.random.default_rng(4)
    keep = []
    descs = []
    for _ in range(2):
        (ci, pj, cj), val = random_dcsr(rng, 5000, 3000, 0.01)
        descs.append(_lib.DcsrDesc(5000, 3000, len(ci), _dev(gpu, keep, ci), _dev(gpu, keep, pj),
                                   len(cj), _dev(gpu, keep, cj), _dev(gpu, keep, val), len(val)))
    return "nacho_gpu_dcsr_mul_f32", descs, _lib.DcsrDesc, keep


@pytest.mark.parametrize("product", ["sssmm", "spgemm", "dcsr_mul"])
def test_call_after_a_failed_allocation(gpu, product):
    entry, descs, result, keep = {"sssmm": _sssmm, "spgemm": _spgemm,
                                  "dcsr_mul": _dcsr_mul}[product](gpu)
    rc, whole, _ = _call(gpu, entry, descs, result, 0)
    torch.cuda.synchronize()
    assert rc == 0 and whole.requests > 5

    rng = np.random.default_rng(1)
    a, b, c = (random_csr(rng, 60, 60, 0.1) for _ in range(3))
    da, db = (random_dcsr(rng, 70, 50, 0.1) for _ in range(2))
    for fail_at in range(1, whole.requests + 1):
        print(f"[gpu] {product}: request {fail_at} of {whole.requests} fails", flush=True)
        torch.cuda._sleep(2_000_000)  # what the call queues stays queued while it fails
        rc, alloc, z = _call(gpu, entry, descs, result, fail_at)
        assert rc == -3, rc
        assert not alloc.held
        assert all(not getattr(z, f) for f, _ in result._fields_)
        if product == "sssmm":
            check_sssmm(run_sssmm(a, b, c, ((60, 60),) * 3, gpu),
                        oracle.port_sssmm(60, 60, a, b, c), f"after {fail_at}")
        elif product == "spgemm":
            run_and_check(gpu, 60, 60, 60, a, b, f"after {fail_at}")
        else:
            assert_dcsr_equal(run_dcsr("mul", (70, 50), da, db, gpu),
                              want_dcsr("mul", da, db), f"after {fail_at}")
    del keep


@pytest.mark.parametrize("polls", [1, 2, 20])
def test_a_tile_that_gives_up(gpu, polls):
    """One-launch levels whose workgroups look only a few times for the counts before theirs: a
    call fails or its result is whole, and the calls after it are correct."""
    import nacho_amd
    from nacho_amd import _lib
    from tests.helpers import assert_csr_equal
    from tests.test_gpu_csr import from_gpu, to_gpu

    rng = np.random.default_rng(polls)
    rows = cols = 20_000
    t = []
    for _ in range(2):
        keys = np.unique(rng.integers(0, rows * cols, size=8 * rows))
        pos = np.concatenate([[0], np.cumsum(np.bincount(keys // cols, minlength=rows))])
        t.append((pos.astype(np.int32), (keys % cols).astype(np.int32),
                  rng.uniform(-1, 1, len(keys)).astype(np.float32)))
    want = oracle.closed_csr_binary("add", rows, cols, *t[0], *t[1])
    a, b = (to_gpu(x, rows, cols, gpu) for x in t)
    lib = _lib.load()
    failed = 0
    try:
        lib.nacho_set_wait_limit(polls)
        for call in range(30):
            print(f"[gpu] at most {polls} polls, call {call}", flush=True)
            try:
                z = nacho_amd.gpu_csr_add_f32(a, b)
            except RuntimeError as e:
                assert "internal" in str(e)
                failed += 1
                continue
            assert_csr_equal(from_gpu(z), want, f"call {call}")
    finally:
        lib.nacho_set_wait_limit(0)
    if polls == 1:
        assert failed, "no wait ended early"
    for call in range(3):
        assert_csr_equal(from_gpu(nacho_amd.gpu_csr_add_f32(a, b)), want, f"after, call {call}")
