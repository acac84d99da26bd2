"""The framework's workloads as timed cases: which entry point, on which operands.

A case names one `gpu_<kernel>_f32` entry point and the operands it meets: row lengths or
fibres drawn from a Zipf law (graphs, web and interaction data) or spread evenly (meshes,
stencils, generated .mtx files), R-MAT graphs for the products, and order-3 tensors with a
Zipf first mode.  The formulas are those of nacho_amd/synth.py, drawn on the GPU so that new
inputs take milliseconds.  Coordinates are sorted and distinct, values uniform.

A case's sizes, those of its results among them, are the same for every seed: one pattern is
drawn per case, and the seed renames its rows, columns, modes or vertices and draws the
values.  Rows and columns that are drawn alike are renamed at random; a tensor's first mode
keeps its order (Zipf ranks), and an R-MAT graph's vertices are renamed by exclusive or, which
only swaps quadrants.
"""

import math

import numpy as np
import torch

import nacho_amd

DEVICE = "cuda"

# Products (a_ij, b_jk pairs) past which exact() would take too long.
MAX_EXACT_PRODUCTS = 1.5e9

MATRIX_OPS = ("csr_add", "csr_add_3", "csr_mul", "coo_add", "coo_mul", "coo_csr_add",
              "dcsr_add", "dcsr_mul")
TENSOR_OPS = ("coo3d_add", "csf_add", "inner_prod", "inner_prod_coo")
PRODUCT_OPS = ("spgemm", "spgemm64", "sssmm")


def listed():
    return [
        # The reference's smoke-test matrices: the smallest call, all latency.
        {"name": "csr_add_smoke", "op": "csr_add", "rows": 200, "cols": 180, "mean": 9.0,
         "lengths": "uniform", "shared": 0.0},
        # C1: a small sparse update, still a launch-bound call.
        {"name": "csr_mul_4096", "op": "csr_mul", "rows": 4096, "cols": 4096, "mean": 41.0,
         "lengths": "uniform", "shared": 0.5},
        # C2: the headline addition, power-law rows.
        {"name": "csr_add_zipf", "op": "csr_add", "rows": 1 << 20, "cols": 1 << 20,
         "mean": 16.0, "lengths": "zipf", "shared": 0.0},
        # Two mesh-like matrices clipped to a common odd shape (the .mtx workload).
        {"name": "csr_add_uniform", "op": "csr_add", "rows": 949_999, "cols": 1_000_003,
         "mean": 8.2, "lengths": "uniform", "shared": 0.0},
        # C3: masking one matrix by another that shares half of it.
        {"name": "csr_mul_overlap", "op": "csr_mul", "rows": 1 << 20, "cols": 1 << 20,
         "mean": 16.0, "lengths": "zipf", "shared": 0.5},
        # Three C2 operands summed in one call.
        {"name": "csr_add_3_zipf", "op": "csr_add_3", "rows": 1 << 20, "cols": 1 << 20,
         "mean": 16.0, "lengths": "zipf", "shared": 0.0},
        # C5 as coordinate lists and as a compressed fibre tree.
        {"name": "coo3d_add_zipf", "op": "coo3d_add", "i": 200_000, "j": 100_000, "k": 1_000,
         "entries": 20_000_000, "shared": 0.0},
        {"name": "csf_add_zipf", "op": "csf_add", "i": 200_000, "j": 100_000, "k": 1_000,
         "entries": 20_000_000, "shared": 0.0},
        # The inner product of two C5 tensors (a decomposition's fit).
        {"name": "inner_prod_zipf", "op": "inner_prod", "i": 200_000, "j": 100_000,
         "k": 1_000, "entries": 20_000_000, "shared": 0.0},
        # Two-hop neighbourhoods of an ordinary graph.
        {"name": "spgemm_rmat13", "op": "spgemm", "graph": "rmat", "scale": 13, "mean": 8.0},
        # C4: the same for a large one; its result needs 64-bit offsets.
        {"name": "spgemm_rmat20", "op": "spgemm64", "graph": "rmat", "scale": 20, "mean": 8.0},
        # Triangle counting on the large graph: the product masked by the graph itself.
        {"name": "sssmm_rmat20", "op": "sssmm", "graph": "rmat", "scale": 20, "mean": 8.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(MATRIX_OPS + TENSOR_OPS + PRODUCT_OPS)
    if op in MATRIX_OPS:
        rows, cols = _log_int(rng, 100, 1 << 20), _log_int(rng, 100, 1 << 20)
        mean = math.exp(rng.uniform(math.log(1.0), math.log(min(64.0, cols / 8))))
        mean = min(mean, 16.0 * (1 << 20) / rows)
        shared = 0.5 if op in ("csr_mul", "coo_mul", "dcsr_mul") else rng.choice((0.0, 0.25))
        return {"op": op, "rows": rows, "cols": cols, "mean": round(mean, 3),
                "lengths": rng.choice(("zipf", "uniform")), "shared": shared}
    if op in TENSOR_OPS:
        i, j, k = _log_int(rng, 50, 200_000), _log_int(rng, 50, 100_000), _log_int(rng, 20, 1_000)
        entries = min(_log_int(rng, 1 << 10, 20_000_000), max(1000, i * j * k // 8))
        shared = rng.choice((0.0, 0.25)) if op in ("coo3d_add", "csf_add") else 0.25
        return {"op": op, "i": i, "j": j, "k": k, "entries": entries, "shared": shared}
    if rng.random() < 0.5:
        return {"op": op, "graph": "rmat", "scale": rng.randint(8, 18),
                "mean": round(rng.uniform(4.0, 9.0), 3)}
    return {"op": op, "graph": "uniform", "rows": _log_int(rng, 100, 300_000),
            "mean": round(rng.uniform(3.0, 20.0), 3)}


# ---- operands ------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _pattern_generator(which):
    return _generator(1 + which)  # operand A from 1, B from 2, as the benchmark's


def _renamed(g, n):
    return torch.randperm(n, generator=g, device=DEVICE)


def _values(g, n, lo=-1.0, hi=1.0):
    return torch.rand(n, generator=g, device=DEVICE) * (hi - lo) + lo


def _lengths(g, case):
    """Entries per row: even (Poisson-like) or a capped Zipf(1.6) rescaled to the mean."""
    rows, cols, mean = case["rows"], case["cols"], case["mean"]
    cap = min(65536, cols // 4)
    if case["lengths"] == "uniform":
        return torch.poisson(torch.full((rows,), mean, device=DEVICE), generator=g).long() \
            .clamp_(0, cols // 2)
    pmf = torch.arange(1, 65537, device=DEVICE, dtype=torch.float64) ** -1.6
    zeta = float(torch.special.zeta(torch.tensor(1.6, dtype=torch.float64),
                                    torch.tensor(1.0, dtype=torch.float64)))
    cdf = (pmf / zeta).cumsum(0)
    u = torch.rand(rows, generator=g, device=DEVICE, dtype=torch.float64)
    raw = (torch.searchsorted(cdf, u) + 1).clamp_(max=65536).double()
    return (raw * (mean * rows / raw.sum())).round_().long().clamp_(0, cap)


def _fresh_keys(g, lengths, cols):
    row = torch.repeat_interleave(torch.arange(len(lengths), device=DEVICE), lengths)
    return row * cols + torch.randint(cols, (len(row),), generator=g, device=DEVICE)


def _share(g, first, fresh, shared):
    """Sorted distinct keys: each of `first` with probability `shared`, the rest fresh."""
    if not shared:
        return torch.unique(fresh)
    kept = first[torch.rand(len(first), generator=g, device=DEVICE) < shared]
    fresh = fresh[torch.rand(len(fresh), generator=g, device=DEVICE) >= shared]
    return torch.unique(torch.cat((kept, fresh)))


def _matrix_keys(case, seed):
    """Each operand's sorted keys row * cols + column, and its values."""
    rows, cols = case["rows"], case["cols"]
    patterns, lengths = [], None
    for which in range(3 if case["op"] == "csr_add_3" else 2):
        g = _pattern_generator(which)
        if lengths is None or not case["shared"]:  # operands that share entries share rows
            lengths = _lengths(g, case)
        fresh = _fresh_keys(g, lengths, cols)
        patterns.append(_share(g, patterns[0] if patterns else None, fresh,
                               case["shared"] if which else 0.0))
    g = _generator(seed)
    row, col = _renamed(g, rows), _renamed(g, cols)
    keys = [torch.sort(row[p // cols] * cols + col[p % cols])[0] for p in patterns]
    return keys, [_values(g, len(k)) for k in keys]


def _tensor_keys(case, seed):
    """Each operand's sorted keys (i * J + j) * K + k, and its values."""
    nj, nk = case["j"], case["k"]
    patterns = []
    cdf = (torch.arange(1, case["i"] + 1, device=DEVICE, dtype=torch.float64) ** -1.3).cumsum(0)
    for which in range(2):
        g = _pattern_generator(which)
        n = case["entries"]
        u = torch.rand(n, generator=g, device=DEVICE, dtype=torch.float64) * cdf[-1]
        i = torch.searchsorted(cdf, u).clamp_(max=case["i"] - 1)
        fresh = (i * nj + torch.randint(nj, (n,), generator=g, device=DEVICE)) * nk \
            + torch.randint(nk, (n,), generator=g, device=DEVICE)
        patterns.append(_share(g, patterns[0] if patterns else None, fresh,
                               case["shared"] if which else 0.0))
    g = _generator(seed)
    j, k = _renamed(g, nj), _renamed(g, nk)
    keys = [torch.sort((p // (nj * nk) * nj + j[p // nk % nj]) * nk + k[p % nk])[0]
            for p in patterns]
    # Counts and ratings for the inner products (no cancellation), signed for the sums.
    lo = 0.0 if case["op"].startswith("inner") else -1.0
    return keys, [_values(g, len(k), lo) for k in keys]


def _graph(case, seed):
    """A graph's adjacency: vertices, sorted keys row * n + column, values in [0.5, 1.5]."""
    g, named = _pattern_generator(0), _generator(seed)
    if case["graph"] == "rmat":
        n = 1 << case["scale"]
        edges = int(case["mean"] * n)
        row = torch.zeros(edges, dtype=torch.int64, device=DEVICE)
        col = torch.zeros(edges, dtype=torch.int64, device=DEVICE)
        for _ in range(case["scale"]):  # quadrant probabilities .57, .19, .19, .05
            r = torch.rand(edges, generator=g, device=DEVICE)
            row = (row << 1) | (r >= 0.76)
            col = (col << 1) | (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        mask = torch.randint(n, (1,), generator=named, device=DEVICE)
        keys = torch.unique((row ^ mask) * n + (col ^ mask))
    else:
        n = case["rows"]
        keys = torch.randint(n * n, (int(case["mean"] * n),), generator=g, device=DEVICE)
        vertex = _renamed(named, n)
        keys = torch.unique(vertex[keys // n] * n + vertex[keys % n])
    return n, keys, _values(named, len(keys), 0.5, 1.5)


def _pos(ids, count):
    """Offsets of each of `count` groups in the sorted group ids `ids`."""
    pos = torch.zeros(count + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(torch.bincount(ids, minlength=count), 0, out=pos[1:])
    return pos


def _int(t):
    return t.to(torch.int32).contiguous()


def _shape(*sizes):
    return torch.tensor(sizes, dtype=torch.int32)


def _csr_arrays(keys, rows, cols):
    return {"pos": _pos(keys // cols, rows), "crd": keys % cols}


def _dcsr_arrays(keys, cols):
    crd_i, counts = torch.unique_consecutive(keys // cols, return_counts=True)
    return {"crd_i": crd_i, "pos": torch.nn.functional.pad(counts.cumsum(0), (1, 0)),
            "crd": keys % cols}


def _csf_arrays(keys, j, k):
    ij, counts_k = torch.unique_consecutive(keys // k, return_counts=True)
    crd_i, counts_j = torch.unique_consecutive(ij // j, return_counts=True)
    return {"crd_i": crd_i, "pos_j": torch.nn.functional.pad(counts_j.cumsum(0), (1, 0)),
            "crd_j": ij % j, "pos_k": torch.nn.functional.pad(counts_k.cumsum(0), (1, 0)),
            "crd_k": keys % k}


def _arrays(kind, keys, case):
    """The level arrays of one operand or result, in the format `kind`."""
    if kind == "csr":
        return _csr_arrays(keys, case["rows"], case["cols"])
    if kind == "coo":
        return {"crd_i": keys // case["cols"], "crd": keys % case["cols"]}
    if kind == "dcsr":
        return _dcsr_arrays(keys, case["cols"])
    if kind == "csf":
        return _csf_arrays(keys, case["j"], case["k"])
    return {"crd_i": keys // (case["j"] * case["k"]), "crd_j": keys // case["k"] % case["j"],
            "crd_k": keys % case["k"]}


# The operands' formats and the result's, by entry point.
_KINDS = {
    "csr_add": ("csr", "csr", "csr"), "csr_add_3": ("csr", "csr", "csr"),
    "csr_mul": ("csr", "csr", "csr"), "coo_add": ("coo", "coo", "coo"),
    "coo_mul": ("coo", "coo", "coo"), "coo_csr_add": ("csr", "coo", "csr"),
    "dcsr_add": ("dcsr", "dcsr", "dcsr"), "dcsr_mul": ("dcsr", "dcsr", "dcsr"),
    "coo3d_add": ("coo3", "coo3", "coo3"), "csf_add": ("csf", "csf", "csf"),
    "inner_prod": ("csf", "csf", "scalar"), "inner_prod_coo": ("coo3", "coo3", "scalar"),
}
_CLASSES = {"csr": nacho_amd.CSR_gpu, "coo": nacho_amd.COO_gpu, "dcsr": nacho_amd.DCSR_gpu,
            "csf": nacho_amd.CSF3_gpu, "coo3": nacho_amd.COO3_gpu}
_FIELDS = {"pos": "dim_j_offsets", "crd": "dim_j_indices", "crd_i": "dim_i_indices",
           "crd_j": "dim_j_indices", "crd_k": "dim_k_indices", "pos_j": "dim_j_offsets",
           "pos_k": "dim_k_offsets", "val": "values"}
_RESULTS = {"csr": ("pos", "crd", "val"), "coo": ("crd_i", "crd", "val"),
            "dcsr": ("crd_i", "pos", "crd", "val"),
            "csf": ("crd_i", "pos_j", "crd_j", "pos_k", "crd_k", "val"),
            "coo3": ("crd_i", "crd_j", "crd_k", "val"), "scalar": ("val",)}


def _keys(case, seed):
    return (_matrix_keys if case["op"] in MATRIX_OPS else _tensor_keys)(case, seed)


def prepare(case, seed):
    op = case["op"]
    call = getattr(nacho_amd, f"gpu_{op}_f32")
    if op in PRODUCT_OPS:
        n, keys, values = _graph(case, seed)
        a = nacho_amd.CSR_gpu(*(_int(t) for t in _csr_arrays(keys, n, n).values()), values,
                              _shape(n, n))
        return {"call": call, "operands": (a,) * (3 if op == "sssmm" else 2), "kind": "csr"}
    shape = _shape(case["rows"], case["cols"]) if op in MATRIX_OPS else \
        _shape(case["i"], case["j"], case["k"])
    operands = []
    for which, (keys, values) in enumerate(zip(*_keys(case, seed))):
        kind = _KINDS[op][min(which, 1)]
        arrays = (_int(t) for t in _arrays(kind, keys, case).values())
        operands.append(_CLASSES[kind](*arrays, values, shape))
    return {"call": call, "operands": tuple(operands), "kind": _KINDS[op][2]}


def run(state):
    z = state["call"](*state["operands"])
    return {name: getattr(z, _FIELDS[name]) for name in _RESULTS[state["kind"]]}


# ---- what the path cannot do without -------------------------------------------------

def _distinct_fibres(case):
    """Expected (i, j) fibres of one operand."""
    p = np.arange(1, case["i"] + 1, dtype=np.float64) ** -1.3
    expected = case["entries"] * p / p.sum()
    return float((case["j"] * -np.expm1(-expected / case["j"])).sum())


def _graph_sizes(case):
    """Expected (vertices, entries, products) of one graph squared."""
    if case["graph"] == "uniform":
        n = case["rows"]
        return n, case["mean"] * n, case["mean"] ** 2 * n
    n = 1 << case["scale"]
    entries = case["mean"] * n
    # Duplicate edges (a few percent of the entries) touch hubs twice: 0.75 of the products
    # that independent edges would give, measured from scale 13 to 20.
    return n, entries, 0.75 * entries ** 2 * (0.76 ** 2 + 0.24 ** 2) ** case["scale"]


def work(case):
    """Every array of the operands and of the result once, at the expected sizes; one
    operation per stored result (per product for the products)."""
    op = case["op"]
    if op in PRODUCT_OPS:
        n, entries, products = _graph_sizes(case)
        if op == "sssmm":
            return {"bytes": 16 * n + 4 * 8 * entries, "flops": 3 * min(products, 16 * entries)}
        # 0.6 distinct outputs per product at scale 20, about as many at the others.
        return {"bytes": 2 * (4 * n + 8 * entries) + 8 * n + 8 * 0.6 * products,
                "flops": 2 * products}
    if op in MATRIX_OPS:
        entries = case["mean"] * case["rows"]
        shared = entries * max(case["shared"], case["mean"] / case["cols"])
        operands = 3 if op == "csr_add_3" else 2
        out = shared if op.endswith("mul") else operands * entries - (operands - 1) * shared
        per_row = {"csr": 4 * case["rows"], "coo": 0, "dcsr": 8 * min(case["rows"], entries)}
        per_entry = {"csr": 8, "coo": 12, "dcsr": 8}
        ka, kb, kz = _KINDS[op]
        total = sum(per_row[k] + per_entry[k] * m for k, m in
                    ((ka, entries), (kb, (operands - 1) * entries), (kz, out)))
        return {"bytes": total + (operands - 2) * per_row[kb], "flops": out}
    entries = case["entries"]
    shared = entries * case["shared"]
    out = 2 * entries - shared
    if _KINDS[op][0] == "coo3":
        return {"bytes": 32 * entries + (16 * out if op == "coo3d_add" else 4),
                "flops": out if op == "coo3d_add" else 2 * entries}
    fibres = _distinct_fibres(case)
    total = 2 * (8 * min(case["i"], fibres) + 8 * fibres + 8 * entries)
    if op == "csf_add":
        total += 8 * case["i"] + 8 * min(2 * fibres, out) + 8 * out
    return {"bytes": total, "flops": out if op == "csf_add" else 2 * entries}


def tolerance(case):
    op = case["op"]
    if op in ("inner_prod", "inner_prod_coo"):
        # Products of one sign, each rounded to float32: 2e-8 off from 64 bits at most in
        # every size measured; sums kept in 32 bits per block show a few 1e-7.
        return {"rel": 1e-6}
    if op in PRODUCT_OPS:
        # Positive float32 products, one more float32 rounding per stored value: 2.7e-8 off
        # from 64 bits (measured at scale 13), the same in any order.
        return {"rel": 1.2e-7, "max": 5e-7}
    return "exact"  # one float32 operation per value (two, in a fixed order, for three)


# ---- the same in 64 bits -------------------------------------------------------------

def _exact_products(case, seed):
    """A * A by expanding row blocks in float64; masked by A for sssmm."""
    n, keys, values = _graph(case, seed)
    row, col, values = keys // n, keys % n, values.double()
    pos = _pos(row, n)
    lengths = (pos[1:] - pos[:-1])[col]
    ends = lengths.cumsum(0)
    if float(ends[-1]) > MAX_EXACT_PRODUCTS:
        return None
    masked = case["op"] == "sssmm"
    out_keys, out_values = [], []
    total = torch.zeros(len(keys), dtype=torch.float64, device=DEVICE)
    reached = torch.zeros(len(keys), dtype=torch.bool, device=DEVICE)
    begin, limit = 0, 1 << 26
    host_ends, host_pos = ends.cpu().numpy(), pos.cpu().numpy()
    while begin < n:  # rows [begin, end): at most `limit` products, or one row
        first = host_pos[begin]
        done = host_ends[first - 1] if first else 0
        entry = np.searchsorted(host_ends, done + limit, side="right")
        end = max(begin + 1, int(np.searchsorted(host_pos, entry, side="right")) - 1)
        last = host_pos[end]
        span = lengths[first:last]
        e = torch.repeat_interleave(torch.arange(first, last, device=DEVICE), span)
        b = torch.arange(len(e), device=DEVICE) - (ends[e] - lengths[e] - done) + pos[col[e]]
        k = row[e] * n + col[b]
        v = values[e] * values[b]
        if masked:
            at = torch.searchsorted(keys, k).clamp_(max=len(keys) - 1)
            hit = keys[at] == k
            total.index_add_(0, at[hit], v[hit] * values[at[hit]])
            reached[at[hit]] = True
        elif len(k):
            k, where = torch.unique(k, return_inverse=True)
            out_keys.append(k)
            out_values.append(torch.zeros(len(k), dtype=torch.float64, device=DEVICE)
                              .index_add_(0, where, v))
        begin = end
    if masked:
        out, val = keys[reached], total[reached]
    else:
        empty = torch.zeros(0, device=DEVICE)
        out, val = torch.cat(out_keys or [empty.long()]), torch.cat(out_values or [empty.double()])
    return {**_csr_arrays(out, n, n), "val": val}


def exact(case, seed):
    if case["op"] in PRODUCT_OPS:
        return _exact_products(case, seed)
    keys, values = _keys(case, seed)
    values = [v.double() for v in values]
    kind = _KINDS[case["op"]][2]
    if kind == "scalar" or case["op"].endswith("mul"):
        at = torch.searchsorted(keys[1], keys[0]).clamp_(max=max(len(keys[1]) - 1, 0))
        hit = keys[1][at] == keys[0]
        out, val = keys[0][hit], values[0][hit] * values[1][at[hit]]
        if kind == "scalar":
            return {"val": val.sum().reshape(1)}
        arrays = _arrays(kind, out, case)
        if kind == "dcsr":  # a row stored in both operands stays, also without a common entry
            rows = [torch.unique_consecutive(k // case["cols"]) for k in keys]
            crd_i = rows[0][torch.isin(rows[0], rows[1])]
            counts = torch.bincount(out // case["cols"], minlength=case["rows"])[crd_i]
            arrays.update(crd_i=crd_i, pos=torch.nn.functional.pad(counts.cumsum(0), (1, 0)))
        return {**arrays, "val": val}
    out = torch.unique(torch.cat(keys))
    val = torch.zeros(len(out), dtype=torch.float64, device=DEVICE)
    for k, v in zip(keys, values):
        val[torch.searchsorted(out, k)] += v
    return {**_arrays(kind, out, case), "val": val}
