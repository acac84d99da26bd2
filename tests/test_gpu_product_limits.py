"""The products' size rules at their limits: scans of up to four chunks of 4096 in one launch, of
up to 2048 in two and longer ones in three, SpGEMM with and without long rows and past the run
count that is bounded instead of counted (2^22 products), sssmm chunks of more mask entries than
keep their fields and sums in LDS (256)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle
from tests.helpers import csr_from_rows, random_csr
from tests.test_gpu_spgemm import run_and_check, spgemm
from tests.test_gpu_sssmm import check as check_sssmm
from tests.test_gpu_sssmm import run as run_sssmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [4095, 4096, 4097, 16383, 16384, 16385, 20481])
def test_scans_at_chunk_limits(gpu, rows):
    rng = np.random.default_rng(rows)
    a = random_csr(rng, rows, 64, 0.02)
    b = random_csr(rng, 64, 500, 0.05)
    run_and_check(gpu, rows, 64, 500, a, b, f"{rows} rows")


@pytest.mark.parametrize("chunks,more", [(2048, 0), (2048, 1), (2049, 4095), (3100, 7)])
def test_scans_of_many_chunks(gpu, chunks, more):
    """Either side of the 2048 chunks whose sums a chunk adds up itself: rows of A with one entry
    or none, B rows of 0 to 2 entries."""
    rng = np.random.default_rng(chunks + more)
    rows, inner = chunks * 4096 + more, 1000
    pos = np.zeros(rows + 1, np.int64)
    np.cumsum(rng.random(rows) < 0.25, out=pos[1:])
    crd = rng.integers(0, inner, pos[-1]).astype(np.int32)
    a = (pos.astype(np.int32), crd, rng.uniform(0.5, 1.5, len(crd)).astype(np.float32))
    len_b = rng.integers(0, 3, inner)
    pos_b = np.concatenate([[0], np.cumsum(len_b)]).astype(np.int32)
    crd_b = np.concatenate([np.sort(rng.choice(50, n, replace=False)) for n in len_b])
    b = (pos_b, crd_b.astype(np.int32), rng.uniform(-1, 1, len(crd_b)).astype(np.float32))
    got = spgemm(a, b, rows, inner, 50, gpu)
    n = len_b[crd]  # a row's result is its one B row, scaled
    want_pos = np.concatenate([[0], np.cumsum(n)])[pos]
    assert np.array_equal(got[0], want_pos)
    at = np.repeat(pos_b[crd] - np.concatenate([[0], np.cumsum(n)[:-1]]), n) + np.arange(n.sum())
    assert np.array_equal(got[1], b[1][at])
    assert np.array_equal(got[2], np.repeat(a[2], n) * b[2][at])


@pytest.mark.parametrize("long_rows", [0, 1, 3])
def test_with_and_without_long_rows(gpu, long_rows):
    """Rows of at most 20 products, and `long_rows` rows of 2500 among them."""
    rng = np.random.default_rng(long_rows)
    n = 600
    rows_a = [[int(r) % n, (int(r) * 7 + 1) % n] for r in range(n)]
    rows_a = [sorted(set(r)) for r in rows_a]
    for i in range(long_rows):
        rows_a[100 * i + 50] = list(range(0, n, 2))
    nnz_a = sum(len(r) for r in rows_a)
    a = csr_from_rows(n, n, rows_a, rng.uniform(0.5, 1.5, nnz_a).astype(np.float32))
    b = random_csr(rng, n, 40000, 9 / 40000)
    run_and_check(gpu, n, n, 40000, a, b, f"{long_rows} long rows")


@pytest.mark.parametrize("copies", [1, 4])
@pytest.mark.parametrize("empty", [0, 60_000])
def test_rows_of_a_by_length(gpu, copies, empty):
    """A's rows on both sides of what a lane group takes (64), of the spans (4096) that long rows are
    split into and of several of those, side by side; with and without the split (32,768 entries)
    and, with many empty rows, one lane per row."""
    rng = np.random.default_rng(copies + empty)
    inner = 24_000
    lengths = np.array([0, 1, 8, 9, 63, 64, 65, 66, 127, 500, 700, 4095, 4096, 4097, 9000] * copies
                       + [20_000] * (copies > 1) + [0] * empty + [2] * 300)
    if empty:
        lengths = rng.permutation(lengths)
    rows_a = [np.sort(rng.choice(inner, size=n, replace=False)).tolist() for n in lengths]
    a = csr_from_rows(len(lengths), inner, rows_a,
                      rng.uniform(0.5, 1.5, int(lengths.sum())).astype(np.float32))
    rows_b = [np.sort(rng.choice(700, size=int(n), replace=False)).tolist()
              for n in rng.integers(0, 4, inner)]
    nnz_b = sum(len(r) for r in rows_b)
    b = csr_from_rows(inner, 700, rows_b, rng.uniform(-1, 1, nnz_b).astype(np.float32))
    run_and_check(gpu, len(lengths), inner, 700, a, b, f"{copies} copies, {empty} empty rows")


@pytest.mark.parametrize("length", [2047, 2049])
def test_runs_bounded_and_counted(gpu, length):
    """2048 rows of `length` products: either side of 2^22 products."""
    rng = np.random.default_rng(length)
    n = 2048
    a = csr_from_rows(n, n, [[i] for i in range(n)], rng.uniform(0.5, 1.5, n).astype(np.float32))
    rows_b = [np.sort(rng.choice(8192, size=length, replace=False)).tolist() for _ in range(n)]
    b = csr_from_rows(n, 8192, rows_b, rng.uniform(-1, 1, n * length).astype(np.float32))
    run_and_check(gpu, n, n, 8192, a, b, f"rows of {length}")


@pytest.mark.parametrize("probes", [1, 15, 16, 17, 300])
def test_sssmm_entries_per_chunk(gpu, probes):
    """Mask entries of `probes` probes each: 4096, 273, 256, 241 and 14 entries per chunk of
    4096 probes."""
    rng = np.random.default_rng(probes)
    n, inner = 120, 400
    rows_a = [np.sort(rng.choice(inner, size=probes, replace=False)).tolist() for _ in range(n)]
    a = csr_from_rows(n, inner, rows_a, rng.uniform(0.5, 1.5, n * probes).astype(np.float32))
    b = random_csr(rng, inner, 100, 0.9)  # columns longer than the rows of A
    c = random_csr(rng, n, 100, 0.8)
    check_sssmm(run_sssmm(a, b, c, ((n, inner), (inner, 100), (n, 100)), gpu),
                oracle.port_sssmm(n, 100, a, b, c), f"{probes} probes")


@pytest.mark.parametrize("half", [0, 1, 2, 7, 8, 12, 40, "ragged"])
@pytest.mark.parametrize("shuffled", [False, True])
def test_sssmm_bands(gpu, half, shuffled):
    """Bands: lists of 2 half + 1 entries (ragged: 1 to 15), nearly every probe hits, several lanes
    of a wavefront on one mask entry, whose entries change at any lane; and the same with every
    third mask entry elsewhere (misses among the hits)."""
    rng = np.random.default_rng(7 if half == "ragged" else half)
    n = 3000
    halves = rng.integers(0, 8, n) if half == "ragged" else [half] * n
    rows = [list(range(max(0, i - h), min(n, i + h + 1))) for i, h in enumerate(halves)]
    a, b = (csr_from_rows(n, n, rows, rng.uniform(-1, 1, sum(map(len, rows))).astype(np.float32))
            for _ in range(2))
    mask = rows
    if shuffled:
        mask = [sorted({k if (i + k) % 3 else (k * 7919) % n for k in r})
                for i, r in enumerate(rows)]
    c = csr_from_rows(n, n, mask, rng.uniform(0.5, 1.5, sum(map(len, mask))).astype(np.float32))
    check_sssmm(run_sssmm(a, b, c, ((n, n),) * 3, gpu), oracle.port_sssmm(n, n, a, b, c),
                f"band {half}")
