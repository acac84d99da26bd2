"""SpGEMM units whose products are expanded by windows of 64: run counts around a batch (512
runs) and a mask word (64), product counts around a round (4096), buckets around the products
that a wavefront holds in registers (512) and around the dense rule (1536), runs of one product
and runs longer than a window."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import csr_from_rows
from tests.test_gpu_spgemm import run_and_check

pytestmark = pytest.mark.gpu


def _row_times(rng, lengths, cols, window):
    """A row of len(lengths) entries times B rows of those lengths, each a random subset of the
    column range `window`; a second row repeats the first one's odd entries."""
    m = len(lengths)
    a = csr_from_rows(2, m, [list(range(m)), list(range(1, m, 2))],
                      rng.uniform(0.5, 1.5, m + m // 2).astype(np.float32))
    lo, hi = window
    rows_b = [np.sort(lo + rng.choice(hi - lo, size=n, replace=False)).tolist() for n in lengths]
    b = csr_from_rows(m, cols, rows_b, rng.uniform(-1, 1, sum(lengths)).astype(np.float32))
    return a, b


@pytest.mark.parametrize("runs,length", [(64, 64), (65, 63), (511, 9), (512, 8), (513, 8),
                                         (1025, 4), (4097, 1), (40, 129), (3, 8000), (2100, 1)])
@pytest.mark.parametrize("mode", ["staged", "symbolic"])
def test_dense_units(gpu, monkeypatch, runs, length, mode):
    monkeypatch.setenv("NACHO_SPGEMM_OUTPUT", mode)
    rng = np.random.default_rng(runs * 10 + length)
    a, b = _row_times(rng, [length] * runs, 3 * 8192 + 5, (8192, 2 * 8192))
    run_and_check(gpu, 2, runs, 3 * 8192 + 5, a, b, f"dense {runs}x{length}")


@pytest.mark.parametrize("per_bucket", [1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1535,
                                        1536])
@pytest.mark.parametrize("buckets", [3, 9])
def test_bitmap_units(gpu, per_bucket, buckets):
    """A long row with `per_bucket` products in each of its column buckets but the last, which
    makes the row long; two products on every column."""
    rng = np.random.default_rng(per_bucket + buckets)
    cols = 8192 * (buckets + 1)
    m = 33
    rows_b = [[] for _ in range(m)]
    for bucket in range(buckets):
        for p in range(per_bucket):  # uneven runs, columns in pairs on two rows
            q = p // 2
            rows_b[(q * q + bucket + 3 * (p % 2)) % m].append(bucket * 8192 + (q * 37) % 8192)
    rows_b[0] += list(range(buckets * 8192, buckets * 8192 + 2200))
    rows_b[1] += list(range(buckets * 8192 + 1000, buckets * 8192 + 1500))
    rows_b = [sorted(r) for r in rows_b]
    assert all(len(set(r)) == len(r) for r in rows_b)
    nnz = sum(len(r) for r in rows_b)
    distinct = len(set().union(*rows_b))
    assert nnz == buckets * per_bucket + 2700
    assert distinct == buckets * ((per_bucket + 1) // 2) + 2200
    a = csr_from_rows(2, m, [list(range(m)), list(range(0, m, 3))],
                      rng.uniform(0.5, 1.5, m + (m + 2) // 3).astype(np.float32))
    b = csr_from_rows(m, cols, rows_b, rng.uniform(-1, 1, nnz).astype(np.float32))
    run_and_check(gpu, 2, m, cols, a, b, f"bitmap {per_bucket} in each of {buckets}")
