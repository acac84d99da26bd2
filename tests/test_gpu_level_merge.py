"""The level merge at its limits: tile and wavefront boundaries, 32- and 64-bit merge keys,
sparse tiles (searched) beside dense ones (sorted), empty operands.

Bar: pos / i, crd and values bit-exact against the numpy closed forms, for csr_add / csr_mul
and, through the same levels with output rows, coo_add / coo_mul.
"""

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.helpers import assert_csr_equal, csr_from_rows

pytestmark = pytest.mark.gpu


def _distinct(rng, n, cols):
    """n distinct sorted columns below cols, the last column always among them."""
    c = np.unique(rng.integers(0, cols, size=2 * n + 8))
    c = rng.permutation(c)[: max(n - 1, 0)]
    return np.unique(np.append(c, cols - 1))[-n:] if n else c[:0]


def _partner(rng, c, n, cols):
    """n columns, about half of them out of c."""
    kept = rng.permutation(c)[: n // 2]
    return np.unique(np.append(kept, _distinct(rng, n - len(kept), cols)))


def _case(name):
    rng = np.random.default_rng(7)
    kind, _, arg = name.partition(":")
    if kind == "edge":  # one long row of about half a tile's entries per operand
        n = int(arg)
        c = np.arange(2 * n)
        return 2 * n, [c[::2], c[:0]], [_partner(rng, c[::2], n, 2 * n), c[:3]]
    if kind == "identical":  # pairs across every wavefront boundary, at both parities
        n = int(arg)
        c = np.arange(n)
        return n, [c[:1], c], [c[:0], c]
    if kind == "cols":  # many nearly empty rows beside a long one: the key's row bits
        cols = int(arg)
        a = [_distinct(rng, int(rng.integers(0, 2)), cols) for _ in range(3000)]
        b = [_partner(rng, x, int(rng.integers(0, 2)), cols) for x in a]
        a[1500], b[1500] = _distinct(rng, 900, cols), _distinct(rng, 1100, cols)
        return cols, a, b
    if kind == "few":  # long rows of one operand, `arg` entries of the other in each
        n, cols = int(arg), 1 << 20
        long = [_distinct(rng, 2000, cols) for _ in range(6)]
        short = [_partner(rng, x, n, cols) for x in long]
        a = [long[0], short[1], long[2], [], short[4], long[5]]
        b = [short[0], long[1], short[2], long[3], long[4], []]
        return cols, a, b
    if kind == "gap":  # a tile with more rows than the sparse path takes
        cols, n = 5000, int(arg)
        a = [_distinct(rng, 2500, cols)] + [[]] * n + [_distinct(rng, 2500, cols)]
        b = [[7]] + [[]] * n + [_distinct(rng, 3, cols)]
        return cols, a, b
    raise AssertionError(name)


CASES = (["edge:%d" % n for n in (1, 2015, 2016, 2017, 4031, 4033)] +
         ["identical:%d" % n for n in (1024, 1025, 4031, 9000)] +
         ["cols:%d" % n for n in (1 << 19, (1 << 19) + 1, 1 << 20, 2**31 - 1)] +
         ["few:%d" % n for n in (1, 60, 127, 128, 129, 300)] +
         ["gap:%d" % n for n in (500, 511, 4100)])


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("op", ["add", "mul"])
def test_level_limits(gpu, op, name):
    import nacho_amd

    cols, ra, rb = _case(name)
    rows = len(ra)
    a, b = csr_from_rows(rows, cols, ra), csr_from_rows(rows, cols, rb)
    print(f"[gpu] level merge {op} {name} rows={rows} cols={cols}", flush=True)
    shape = torch.tensor([rows, cols], dtype=torch.int32)

    def dev(x):
        return torch.from_numpy(np.ascontiguousarray(x)).to(gpu)

    want = oracle.closed_csr_binary(op, rows, cols, *a, *b)
    z = getattr(nacho_amd, f"gpu_csr_{op}_f32")(
        *(nacho_amd.CSR_gpu(*(dev(x) for x in t), shape) for t in (a, b)))
    got = tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
    assert_csr_equal(got, want, name)
    row_of = [np.repeat(np.arange(rows, dtype=np.int32), np.diff(t[0])) for t in (a, b, want)]
    z = getattr(nacho_amd, f"gpu_coo_{op}_f32")(
        *(nacho_amd.COO_gpu(dev(i), dev(t[1]), dev(t[2]), shape)
          for i, t in zip(row_of, (a, b))))
    assert np.array_equal(z.dim_i_indices.cpu().numpy(), row_of[2])
    assert np.array_equal(z.dim_j_indices.cpu().numpy(), want[1])
    assert np.array_equal(z.values.cpu().numpy().view(np.uint32), want[2].view(np.uint32))


@pytest.mark.parametrize("op", ["add", "mul"])
@pytest.mark.parametrize("empty", ["a", "b", "both"])
def test_empty_operand(gpu, op, empty):
    import nacho_amd

    c = np.arange(5000)
    full, none = csr_from_rows(2, 5000, [c, c[::3]]), csr_from_rows(2, 5000, [[], []])
    a, b = (none if empty in ("a", "both") else full), (none if empty in ("b", "both") else full)
    shape = torch.tensor([2, 5000], dtype=torch.int32)
    z = getattr(nacho_amd, f"gpu_csr_{op}_f32")(
        *(nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in t), shape) for t in (a, b)))
    got = tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
    assert_csr_equal(got, oracle.closed_csr_binary(op, 2, 5000, *a, *b), empty)


@pytest.mark.parametrize("rows", [1, 230, 245, 500, 60_000, 62_500])
def test_one_launch_limits(gpu, rows):
    """One tile, two, and both sides of the tile count up to which a level is one launch."""
    import nacho_amd

    rng = np.random.default_rng(rows)
    cols = 300_000
    t = []
    for _ in range(2):
        keys = np.unique(rng.integers(0, rows * cols, size=8 * rows))
        pos = np.zeros(rows + 1, np.int32)
        pos[1:] = np.cumsum(np.bincount(keys // cols, minlength=rows))
        t.append((pos, (keys % cols).astype(np.int32),
                  rng.uniform(-1, 1, len(keys)).astype(np.float32)))
    shape = torch.tensor([rows, cols], dtype=torch.int32)
    ops = [nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in o), shape) for o in t]
    for op in ("add", "mul", "add"):  # (the sync block is reused from call to call)
        z = getattr(nacho_amd, f"gpu_csr_{op}_f32")(*ops)
        got = tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
        assert_csr_equal(got, oracle.closed_csr_binary(op, rows, cols, *t[0], *t[1]), op)


def test_one_launch_threads_and_streams(gpu):
    """Threads on one stream and on streams of their own, with the cache given back between."""
    import threading

    import nacho_amd

    rng = np.random.default_rng(3)
    rows = cols = 4000
    t = []
    for _ in range(2):
        keys = np.unique(rng.integers(0, rows * cols, size=40_000))
        pos = np.zeros(rows + 1, np.int32)
        pos[1:] = np.cumsum(np.bincount(keys // cols, minlength=rows))
        t.append((pos, (keys % cols).astype(np.int32),
                  rng.uniform(-1, 1, len(keys)).astype(np.float32)))
    shape = torch.tensor([rows, cols], dtype=torch.int32)
    ops = [nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in o), shape) for o in t]
    torch.cuda.synchronize()
    want = oracle.closed_csr_binary("add", rows, cols, *t[0], *t[1])
    failures = []

    def work(own_stream):
        try:
            stream = torch.cuda.Stream() if own_stream else torch.cuda.default_stream()
            with torch.cuda.stream(stream):
                for i in range(30):
                    z = nacho_amd.gpu_csr_add_f32(*ops)
                    if i % 10 == 9:
                        stream.synchronize()
                        got = tuple(x.cpu().numpy()
                                    for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
                        assert_csr_equal(got, want, f"call {i}")
                        nacho_amd.release_cached_memory()
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=work, args=(k % 2 == 1,)) for k in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failures, failures[0]


def test_one_launch_many_threads(gpu):
    """100 live threads, one call each on one stream: none of them waits for the device (a side
    stream is still busy at the end)."""
    import threading

    import nacho_amd

    rng = np.random.default_rng(5)
    rows, cols = 2000, 3000
    t = [csr_from_rows(rows, cols, [np.unique(rng.integers(0, cols, 8)) for _ in range(rows)])
         for _ in range(2)]
    shape = torch.tensor([rows, cols], dtype=torch.int32)
    ops = [nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in o), shape) for o in t]
    want = oracle.closed_csr_binary("add", rows, cols, *t[0], *t[1])
    main = torch.cuda.Stream()
    begin, end, busy = (torch.cuda.Event(enable_timing=True) for _ in range(3))
    with torch.cuda.stream(main):
        for _ in range(3):  # (warms the buffers up)
            nacho_amd.gpu_csr_add_f32(*ops)
        torch.cuda._sleep(1_000_000)
        begin.record()
        torch.cuda._sleep(1_000_000)
        end.record()
    torch.cuda.synchronize()
    cycles = int(1_000_000 * 300 / begin.elapsed_time(end))  # about 0.3 seconds

    def sleep_on(side):
        with torch.cuda.stream(side):
            torch.cuda._sleep(cycles)
            busy.record()

    # Streams share the few hardware queues of a process: a side stream on another one than main.
    for _ in range(8):
        side = torch.cuda.Stream()
        sleep_on(side)
        with torch.cuda.stream(main):
            nacho_amd.gpu_csr_add_f32(*ops)
        if not busy.query():
            break
        torch.cuda.synchronize()
    else:
        pytest.fail("no stream runs beside the first one")
    torch.cuda.synchronize()
    gates = [threading.Event() for _ in range(101)]
    hold, failures = threading.Event(), []

    def work(i):
        gates[i].wait()
        try:
            with torch.cuda.stream(main):
                nacho_amd.gpu_csr_add_f32(*ops)
        except BaseException as e:  # noqa: BLE001
            failures.append(e)
        gates[i + 1].set()
        hold.wait()  # (a thread that ended would give its id to the next)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(100)]
    for th in threads:
        th.start()
    sleep_on(side)
    gates[0].set()
    gates[100].wait()
    waited = busy.query()
    hold.set()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert not failures, failures[0]
    assert not waited, "a call waited for the device"
    with torch.cuda.stream(main):
        z = nacho_amd.gpu_csr_add_f32(*ops)
    torch.cuda.synchronize()
    assert_csr_equal(tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values)),
                     want, "after")


@pytest.mark.parametrize("lo,hi", [(0, 40), (0, 70_000), (0, 2**31), (-50, 50), (-(2**31), 2**31)])
@pytest.mark.parametrize("rows,mean", [(1, 3000), (40, 400), (3000, 5), (70_000, 12)])
@pytest.mark.parametrize("op", ["add", "mul"])
def test_coordinates_past_the_extent(gpu, op, rows, mean, lo, hi):
    """Coordinates are ordered as the int32 numbers they are, whatever extent is declared (8)."""
    import nacho_amd

    rng = np.random.default_rng(rows + mean)
    n = min(mean, (hi - lo) // 2)
    keys = []
    pool = np.unique(rng.integers(lo, hi, size=4 * n))  # (coordinates that both operands draw)
    for _ in range(2):
        r = np.repeat(np.arange(rows, dtype=np.int64), n)
        keys.append(np.unique(r * 2**33 + pool[rng.integers(0, len(pool), size=len(r))] + 2**32))
    vals = [rng.uniform(-1, 1, len(k)).astype(np.float32) for k in keys]

    def csr(k):
        pos = np.zeros(rows + 1, np.int32)
        pos[1:] = np.cumsum(np.bincount(k >> 33, minlength=rows))
        return pos, ((k & (2**33 - 1)) - 2**32).astype(np.int32)

    both, ia, ib = np.intersect1d(*keys, assume_unique=True, return_indices=True)
    if op == "mul":
        want_keys, want = both, vals[0][ia] * vals[1][ib]
    else:
        want_keys = np.union1d(*keys)
        at = [np.searchsorted(want_keys, k) for k in keys]
        want = np.zeros(len(want_keys), np.float32)
        want[at[1]] = vals[1]
        want[at[0]] = vals[0]
        want[at[0][ia]] = vals[0][ia] + vals[1][ib]
    print(f"[gpu] level merge {op} rows={rows} n={n} coordinates in [{lo}, {hi})", flush=True)
    shape = torch.tensor([rows, 8], dtype=torch.int32)

    def dev(x):
        return torch.from_numpy(np.ascontiguousarray(x)).to(gpu)

    z = getattr(nacho_amd, f"gpu_csr_{op}_f32")(
        *(nacho_amd.CSR_gpu(*(dev(x) for x in csr(k)), dev(v), shape) for k, v in zip(keys, vals)))
    got = tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
    assert_csr_equal(got, (*csr(want_keys), want), op)
    z = getattr(nacho_amd, f"gpu_coo_{op}_f32")(
        *(nacho_amd.COO_gpu(dev((k >> 33).astype(np.int32)), dev(csr(k)[1]), dev(v), shape)
          for k, v in zip(keys, vals)))
    assert np.array_equal(z.dim_i_indices.cpu().numpy(), (want_keys >> 33).astype(np.int32))
    assert np.array_equal(z.dim_j_indices.cpu().numpy(), csr(want_keys)[1])
    assert np.array_equal(z.values.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("na,nb", [(2, 7), (7, 2), (4, 5), (9, 9)])
def test_short_unsorted_rows(gpu, na, nb):
    """Rows whose coordinates are in no order break the contract, but every entry still comes out
    once, in its row (more tiles than one launch takes, few searches in each)."""
    import nacho_amd

    rng = np.random.default_rng(10 * na + nb)
    rows = 160_000
    ca = rng.permuted(np.tile(np.arange(12), (rows, 1)), axis=1)[:, :na] * 2
    cb = rng.permuted(np.tile(np.arange(12), (rows, 1)), axis=1)[:, :nb] * 2 + 1
    # most rows belong to one operand, so that tiles hold few searches
    la = np.where(np.arange(rows) % 16 == 0, na, np.where(np.arange(rows) % 2 == 0, na, 0))
    lb = np.where(np.arange(rows) % 16 == 0, nb, np.where(np.arange(rows) % 2 == 1, nb, 0))
    ops, want = [], []
    for c, n in ((ca, la), (cb, lb)):
        pos = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
        keep = np.arange(c.shape[1])[None, :] < n[:, None]
        crd = c[keep].astype(np.int32)
        val = rng.uniform(-1, 1, len(crd)).astype(np.float32)
        ops.append((pos, crd, val))
        want.append((np.repeat(np.arange(rows), n), crd, val))
    shape = torch.tensor([rows, 24], dtype=torch.int32)
    print(f"[gpu] unsorted rows of {na} and {nb}", flush=True)
    z = nacho_amd.gpu_csr_add_f32(
        *(nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in o), shape) for o in ops))
    pos, crd, val = (x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
    assert np.array_equal(pos, ops[0][0] + ops[1][0])
    row = np.repeat(np.arange(rows), np.diff(pos))
    w = [np.concatenate([x[i] for x in want]) for i in range(3)]
    got, exp = np.lexsort((crd, row)), np.lexsort((w[1], w[0]))
    assert np.array_equal(row[got], w[0][exp]) and np.array_equal(crd[got], w[1][exp])
    assert np.array_equal(val[got], w[2][exp])


@pytest.mark.parametrize("rows,mean", [(50, 30), (90_000, 5), (90_000, 14)])
@pytest.mark.parametrize("op", ["add", "mul"])
def test_arrays_longer_than_the_entries(gpu, op, rows, mean):
    """Coordinate and value arrays with room past the last offset: the result holds the entries
    that the offsets span (in one launch, and in three with and without the sparse split)."""
    import nacho_amd

    rng = np.random.default_rng(mean)
    cols, t = 200_000, []
    for _ in range(2):
        keys = np.unique(rng.integers(0, rows * cols, size=rows * mean))
        pos = np.zeros(rows + 1, np.int32)
        pos[1:] = np.cumsum(np.bincount(keys // cols, minlength=rows))
        t.append((pos, (keys % cols).astype(np.int32),
                  rng.uniform(-1, 1, len(keys)).astype(np.float32)))
    want = oracle.closed_csr_binary(op, rows, cols, *t[0], *t[1])
    room = [(pos, np.append(crd, np.full(777, 5, np.int32)),
             np.append(val, np.full(777, 9, np.float32))) for pos, crd, val in t]
    shape = torch.tensor([rows, cols], dtype=torch.int32)
    print(f"[gpu] {op} rows={rows} mean={mean}, arrays with room", flush=True)
    z = getattr(nacho_amd, f"gpu_csr_{op}_f32")(
        *(nacho_amd.CSR_gpu(*(torch.from_numpy(x).to(gpu) for x in o), shape) for o in room))
    got = tuple(x.cpu().numpy() for x in (z.dim_j_offsets, z.dim_j_indices, z.values))
    assert_csr_equal(got, want, op)
