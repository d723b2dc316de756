"""The calls whose time counts for a user of this library, and their inputs.

Every case is one pass through the public entry points of ``clbool_amd`` on
matrices that are already where a program has them: on the device, except for
the COO construction, whose entry point takes host arrays.  All outputs are
whole numbers (sizes, row pointers, row ids, columns) and are returned whole,
as tensors over the library's own buffers.

Graphs are R-MAT with the usual (.57, .19, .19, .05), duplicates and self-loops
removed, vertex ids below ``n`` (any number, not only a power of two).  A case
has one graph up to its labels: the seed relabels it, so that inputs of
different seeds differ throughout while all sizes, and with them the outputs'
shapes, stay.  R-MAT labels move within aligned groups of 64, which keeps the
generator's locality; uniform and Zipf patterns have none and are relabelled
freely.
"""
import math

import numpy as np
import torch

import clbool_amd as cb
from clbool_amd import generators as gen

QUAD = (0.57, 0.19, 0.19, 0.05)
ZIPF_CAP = 4096
GROUP = 64  # ids that R-MAT labels move among


def listed():
    return [
        # The smallest product in the tests and the README's kind of use: two
        # 1024 x 1024 matrices of 10,000 pairs.  Launches and waits are all of it.
        {"name": "product small", "op": "product", "pattern": "uniform", "mode": "plain",
         "rows": 1024, "inner": 1024, "cols": 1024, "pairs_a": 10000, "pairs_b": 10000},
        # An ordinary product of the drop-in entry point: a graph's two-hop
        # neighbourhood with every row length from one to thousands.
        {"name": "product graph", "op": "product", "pattern": "rmat", "mode": "plain",
         "n": 65536, "edges": 16 * 65536},
        # Hypersparse rows (one in a hundred stored, Zipf lengths) on 2^24
        # columns, sized by the trained predictor: the row map and the
        # many-window columns matter, not the products.
        {"name": "product hypersparse", "op": "product", "pattern": "zipf", "mode": "learned",
         "n": 1 << 24, "row_share": 0.01},
        # The second product of the API (expand, sort, compress) on a graph
        # whose long rows need the global sort; odd sizes.
        {"name": "product sorted", "op": "product", "pattern": "rmat", "mode": "sorted",
         "n": 16001, "edges": 200003},
        # A product larger than its blocks may be, exactly sized, in row blocks.
        {"name": "blocks plain", "op": "blocks", "pattern": "rmat", "mode": "plain",
         "n": 1 << 18, "edges": 16 << 18, "bound": 500_000_000},
        # The benchmark's power-law square at 2^20 vertices by the one pass, in
        # overlapping row blocks: the largest work.
        {"name": "blocks one pass", "op": "blocks", "pattern": "rmat", "mode": "bound",
         "n": 1 << 20, "edges": 16 << 20, "bound": 0},
        # One step of path-query evaluation over 64 labels and 32 rules
        # (X |= Y * Z), all products batched, learned sizing.
        {"name": "closure step", "op": "closure", "mode": "learned", "n": 1 << 18, "labels": 64, "rules": 32,
         "lo": 1 << 10, "hi": 1 << 20},
        # The same with a small grammar on a small graph, where a program
        # calls it many times until nothing changes.
        {"name": "closure step small", "op": "closure", "mode": "plain", "n": 5000, "labels": 6, "rules": 5,
         "lo": 1000, "hi": 20000},
        # The automaton of a regular path query times a graph; both directions
        # of use read its rows afterwards, so it is written whole.
        {"name": "kronecker", "op": "kronecker", "states": 64, "moves": 200, "n": 65536, "edges": 16 * 65536},
        # The union that ends a closure step: a large matrix and a new one, odd sizes.
        {"name": "union", "op": "union", "format": "dcsr", "n": 1000003, "edges_a": 16_000_001,
         "edges_b": 5_000_003},
        # A matrix built from an edge list as it comes from a file: host
        # arrays, unsorted, with duplicates.
        {"name": "construct", "op": "construct", "n": 250007, "edges": 4_000_037},
        # The transposed adjacency of a large graph (backward steps of a traversal).
        {"name": "transpose", "op": "transpose", "n": 1 << 20, "edges": 16 << 20},
    ]


def _log_int(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm, any residue."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["uniform", "graph", "zipf", "sorted", "blocks", "closure", "kronecker", "union", "construct",
                     "transpose"])
    if op == "uniform":
        r, k, c = (_log_int(rng, 300, 30000) for _ in range(3))
        return {"op": "product", "pattern": "uniform", "mode": rng.choice(["plain", "plain", "learned"]),
                "rows": r, "inner": k, "cols": c,
                "pairs_a": min(r * k // 4, r * rng.randint(2, 24)), "pairs_b": min(k * c // 4, k * rng.randint(2, 24))}
    if op == "graph":
        n = _log_int(rng, 2000, 150000)
        return {"op": "product", "pattern": "rmat", "mode": rng.choice(["plain", "plain", "learned"]), "n": n,
                "edges": n * rng.randint(4, 20) + rng.randint(0, 999)}
    if op == "zipf":
        return {"op": "product", "pattern": "zipf", "mode": rng.choice(["plain", "learned"]),
                "n": _log_int(rng, 1 << 20, 1 << 24), "row_share": round(rng.uniform(0.004, 0.012), 4)}
    if op == "sorted":
        n = _log_int(rng, 1000, 20000)
        return {"op": "product", "pattern": "rmat", "mode": "sorted", "n": n,
                "edges": n * rng.randint(4, 12) + rng.randint(0, 999)}
    if op == "blocks":
        mode = rng.choice(["plain", "bound"])
        n = _log_int(rng, 40000, 300000 if mode == "plain" else 800000)
        edges = n * rng.randint(8, 16) + rng.randint(0, 999)
        return {"op": "blocks", "pattern": "rmat", "mode": mode, "n": n,
                "edges": edges, "bound": int(_square_nnz(n, edges, edges)) // rng.randint(1, 6)}
    if op == "closure":
        n = _log_int(rng, 3000, 200000)
        return {"op": "closure", "mode": rng.choice(["plain", "learned"]), "n": n, "labels": rng.randint(4, 48),
                "rules": rng.randint(3, 24), "lo": max(500, n // 256), "hi": min(4 * n, 1 << 19)}
    if op == "kronecker":
        s = rng.randint(3, 64)
        n = _log_int(rng, 1000, 65536)
        return {"op": "kronecker", "states": s, "moves": rng.randint(s, min(s * s // 2, 200)), "n": n,
                "edges": n * rng.randint(3, 16) + rng.randint(0, 999)}
    if op == "union":
        n = _log_int(rng, 1000, 1000000)
        return {"op": "union", "format": rng.choice(["dcsr", "csr", "coo"]), "n": n,
                "edges_a": n * rng.randint(2, 16) + rng.randint(0, 999),
                "edges_b": n * rng.randint(1, 8) + rng.randint(0, 999)}
    n = _log_int(rng, 1000, 250000 if op == "construct" else 1000000)
    return {"op": op, "n": n, "edges": n * rng.randint(3, 16) + rng.randint(0, 999)}


# ---------------------------------------------------------------------------
# What a program has in hand

_kept = {}


def _controls():
    """The one Controls a program keeps."""
    if "controls" not in _kept:
        _kept["controls"] = cb.create_controls(0, 0)
    return _kept["controls"]


def _train(ctl):
    """The predictor, trained once per program on other matrices than the cases'."""
    if "trained" in _kept:
        return
    cb.predictor_reset(ctl, seed=1)
    for scale, factor, seed in ((14, 16, 2), (16, 16, 3)):
        m = cb.matrix_dcsr_from_cpu(ctl, *gen.to_dcsr(*gen.rmat(scale, factor, seed)), 1 << scale)
        cb.predictor_harvest(ctl, m, m)
    for log_n, seed in ((21, 4), (22, 5), (22, 6)):
        m = cb.matrix_dcsr_from_cpu(ctl, *gen.to_dcsr(*gen.hypersparse_zipf(seed, log_n=log_n)), 1 << log_n)
        cb.predictor_harvest(ctl, m, m)
    cb.predictor_train(ctl, epochs=60, batch=1024, lr=2e-3, seed=1)
    _kept["trained"] = True


def _generator(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _relabel(n, group, g):
    """New labels of ids 0..n-1: a random order within aligned groups of ids."""
    ids = torch.arange(n, device="cuda")
    order = torch.argsort((ids // group).double() + torch.rand(n, device="cuda", dtype=torch.float64, generator=g))
    new = torch.empty_like(ids)
    new[order] = ids
    return new


def _moved(keys, new_rows, new_cols):
    """Keys row << 32 | col under new labels (None: the old ones)."""
    row, col = keys >> 32, keys & 0xFFFFFFFF
    return ((row if new_rows is None else new_rows[row]) << 32) | (col if new_cols is None else new_cols[col])


def _rmat_edges(n, edges, which=0):
    """Edges as drawn (int64 keys row << 32 | col): duplicates stay, order random."""
    g = _generator(1000 + which)
    a, b, c, _ = QUAD
    row = torch.zeros(edges, dtype=torch.int64, device="cuda")
    col = torch.zeros_like(row)
    for _ in range(max(1, (n - 1).bit_length())):
        u = torch.rand(edges, device="cuda", generator=g)
        low = u >= a + b
        right = torch.where(low, u >= a + b + c, u >= a)
        row = row * 2 + low
        col = col * 2 + right
    keep = (row != col) & (row < n) & (col < n)
    return ((row << 32) | col)[keep]


def _uniform_edges(rows, cols, pairs, which=0):
    g = _generator(2000 + which)
    cells = torch.unique(torch.randint(0, rows * cols, (pairs + pairs // 4 + 64,), device="cuda", generator=g))
    cells = cells[torch.randperm(cells.numel(), device="cuda", generator=g)[:pairs]]
    return ((cells // cols) << 32) | (cells % cols)


def _zipf_edges(n, row_share):
    """A share of the rows stored, Zipf(1.5) lengths capped at ZIPF_CAP, uniform columns."""
    g = _generator(3000)
    stored = int(n * row_share)
    ids = torch.randperm(n, device="cuda", generator=g)[:stored]
    cdf = torch.tensor(np.cumsum(_zipf_weights()), device="cuda")
    lens = torch.searchsorted(cdf, torch.rand(stored, device="cuda", dtype=torch.float64, generator=g)) + 1
    row = torch.repeat_interleave(ids, lens.clamp(max=ZIPF_CAP))
    return (row << 32) | torch.randint(0, n, (row.numel(),), device="cuda", generator=g)


def _zipf_weights():
    k = np.arange(1, ZIPF_CAP + 1, dtype=np.float64)
    w = k ** -1.5
    w /= 2.612375348685488  # zeta(1.5); the tail beyond the cap goes to the cap
    w[-1] += 1.0 - w.sum()
    return w


def _buffer(ctl, values):
    """A library buffer with a device tensor's values as uint32."""
    b = cb.Buffer.create(ctl, 4 * values.numel())
    _tensor(b, values.numel()).copy_(values.to(torch.int32) if values.dtype != torch.int64 else
                                     (values & 0xFFFFFFFF).to(torch.int32))
    return b


class _Words:
    """A buffer's first n words for torch (which keeps the buffer alive)."""

    def __init__(self, buf, n):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "data": (buf.device_ptr, False),
                                         "strides": None, "version": 3}


def _tensor(buf, n):
    if buf is None or n == 0:
        return torch.empty(0, dtype=torch.int32, device="cuda")
    return torch.as_tensor(_Words(buf, n), device="cuda")


def _dcsr(ctl, keys, nrows, ncols):
    """A matrix_dcsr of the distinct keys row << 32 | col."""
    keys = torch.unique(keys)
    rows, counts = torch.unique_consecutive(keys >> 32, return_counts=True)
    rpt = torch.zeros(rows.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(counts, 0, out=rpt[1:])
    return cb.matrix_dcsr(nrows, ncols, _buffer(ctl, rpt), _buffer(ctl, rows), _buffer(ctl, keys),
                          keys.numel(), rows.numel())


def _csr(ctl, keys, n):
    keys = torch.unique(keys)
    rpt = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(keys >> 32, minlength=n), 0, out=rpt[1:])
    return cb.matrix_csr(n, n, _buffer(ctl, rpt), _buffer(ctl, keys), keys.numel())


def _coo(ctl, keys, n):
    keys = torch.unique(keys)
    return cb.matrix_coo(n, n, _buffer(ctl, keys >> 32), _buffer(ctl, keys), keys.numel())


def _label_sizes(case):
    """Edge counts of the labels: Zipf(1.1) over [lo, hi], in a fixed mixed order."""
    return gen.bounded_zipf_sizes(case["labels"], case["lo"], case["hi"], 1.1, seed=0).tolist()


def _rules(case):
    """The grammar (X, Y, Z label indices): it stays while the graph changes."""
    rng = np.random.default_rng(1)
    heads = min(case["labels"], 20)
    return [(int(rng.integers(0, heads)), int(rng.integers(0, case["labels"])), int(rng.integers(0, case["labels"])))
            for _ in range(case["rules"])]


def prepare(case, seed):
    ctl = _controls()
    g = _generator(seed)
    s = {"case": case, "ctl": ctl}
    op = case["op"]
    if case.get("mode") == "learned":
        _train(ctl)
    n = case.get("n")
    if op == "product" and case["pattern"] == "uniform":
        r, k, c = case["rows"], case["inner"], case["cols"]
        pr, pk, pc = (_relabel(x, x, g) for x in (r, k, c))
        s["a"] = _dcsr(ctl, _moved(_uniform_edges(r, k, case["pairs_a"]), pr, pk), r, k)
        s["b"] = _dcsr(ctl, _moved(_uniform_edges(k, c, case["pairs_b"], 1), pk, pc), k, c)
    elif op == "product" and case["pattern"] == "zipf":
        p = _relabel(n, n, g)
        s["a"] = s["b"] = _dcsr(ctl, _moved(_zipf_edges(n, case["row_share"]), p, p), n, n)
    elif op == "product":
        p = _relabel(n, GROUP, g)
        s["a"] = s["b"] = _dcsr(ctl, _moved(_rmat_edges(n, case["edges"]), p, p), n, n)
    elif op == "blocks":
        # the result's rows keep their order, and with it the blocks' ends
        p, q = _relabel(n, GROUP, g), _relabel(n, GROUP, g)
        keys = _rmat_edges(n, case["edges"])
        s["a"] = _dcsr(ctl, _moved(keys, None, p), n, n)
        s["b"] = _dcsr(ctl, _moved(keys, p, q), n, n)
    elif op == "closure":
        p = _relabel(n, GROUP, g)
        s["mats"] = [_dcsr(ctl, _moved(_rmat_edges(n, m, i), p, p), n, n) for i, m in enumerate(_label_sizes(case))]
        s["rules"] = _rules(case)
    elif op == "kronecker":
        k = case["states"]
        p, q = _relabel(k, k, g), _relabel(n, GROUP, g)
        s["a"] = _dcsr(ctl, _moved(_uniform_edges(k, k, case["moves"]), p, p), k, k)
        s["b"] = _dcsr(ctl, _moved(_rmat_edges(n, case["edges"]), q, q), n, n)
    elif op == "union":
        p = _relabel(n, GROUP, g)
        make = {"dcsr": lambda k: _dcsr(ctl, k, n, n), "csr": lambda k: _csr(ctl, k, n),
                "coo": lambda k: _coo(ctl, k, n)}[case["format"]]
        s["a"] = make(_moved(_rmat_edges(n, case["edges_a"]), p, p))
        s["b"] = make(_moved(_rmat_edges(n, case["edges_b"], 1), p, p))
    elif op == "construct":
        p = _relabel(n, GROUP, g)
        keys = _moved(_rmat_edges(n, case["edges"]), p, p)
        keys = keys[torch.randperm(keys.numel(), device="cuda", generator=g)]
        s["rows"] = (keys >> 32).to(torch.int32).cpu().numpy().view(np.uint32)
        s["cols"] = (keys & 0xFFFFFFFF).to(torch.int32).cpu().numpy().view(np.uint32)
    elif op == "transpose":
        p = _relabel(n, GROUP, g)
        s["a"] = _dcsr(ctl, _moved(_rmat_edges(n, case["edges"]), p, p), n, n)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return s


# ---------------------------------------------------------------------------
# One pass

def _out(m):
    """A matrix's own buffers; its sizes are theirs."""
    if isinstance(m, cb.matrix_dcsr):
        return [_tensor(m.rpt_gpu, m.nzr + 1), _tensor(m.rows_gpu, m.nzr), _tensor(m.cols_gpu, m.nnz)]
    if isinstance(m, cb.matrix_csr):
        return [_tensor(m.rpt_gpu, m.nrows + 1), _tensor(m.cols_gpu, m.nnz)]
    return [_tensor(m.rows_gpu, m.nnz), _tensor(m.cols_gpu, m.nnz)]


MODES = {"plain": cb.SPGEMM_PLAIN, "learned": cb.SPGEMM_LEARNED, "bound": cb.SPGEMM_BOUND}


def run(state):
    case, ctl = state["case"], state["ctl"]
    op = case["op"]
    if op == "product":
        if case["mode"] == "plain":
            return _out(cb.dcsr.matrix_multiplication_hash(ctl, state["a"], state["b"]))
        if case["mode"] == "sorted":
            return _out(cb.dcsr.matrix_multiplication(ctl, state["a"], state["b"]))
        return _out(cb.dcsr.spgemm(ctl, state["a"], state["b"], mode=MODES[case["mode"]])[0])
    if op == "blocks":
        out = []
        plan = cb.dcsr.plan(ctl, state["a"], state["b"], mode=MODES[case["mode"]], block_bound=case["bound"])
        plan.run_all(lambda k, block, stats: out.append(block))
        plan.close()
        return [_out(m) for m in out]
    if op == "closure":
        mats = list(state["mats"])
        cb.closure_step(ctl, mats, state["rules"], mode=cb.CLOSURE_BATCHED, spgemm_mode=MODES[case["mode"]])
        return [_out(mats[x]) for x in sorted({t[0] for t in state["rules"]})]  # what the rules write
    if op == "kronecker":
        return _out(cb.dcsr.kronecker_product(ctl, state["a"], state["b"]))
    if op == "union":
        add = {"dcsr": cb.dcsr.addition, "csr": cb.csr.matrix_addition, "coo": cb.coo.matrix_addition}[case["format"]]
        return _out(add(ctl, state["a"], state["b"]))
    if op == "construct":
        coo = cb.matrix_coo.from_host(ctl, state["rows"], state["cols"], case["n"], case["n"], sorted=False,
                                      noDuplicates=False)
        return _out(cb.coo_to_dcsr_shallow(ctl, coo))
    return _out(cb.dcsr.transpose(ctl, state["a"]))


def exact(case, seed):
    """Every output is a whole number: there is nothing to be nearer to."""
    return None


# ---------------------------------------------------------------------------
# What a pass cannot do without: its inputs read once, its outputs written
# once; one operation per intermediate product.  Sizes are the generators'
# expectations.

def _distinct(levels, weights, draws):
    """Expected distinct cells among `draws` draws (a number) when a cell's share
    is a product of one of the weights per level."""
    total = 0.0
    w = [math.log(x) for x in weights]

    def walk(left, k, cells, logp):
        nonlocal total
        if k == len(w) - 1:
            lam = draws * math.exp(logp + left * w[k])
            total += cells * -math.expm1(-lam)
            return
        for i in range(left + 1):
            walk(left - i, k + 1, cells * math.comb(left, i), logp + i * w[k])

    walk(levels, 0, 1.0, 0.0)
    return total


def _levels(n):
    return max(1, (n - 1).bit_length())


def _rmat_nnz(n, edges):
    return _distinct(_levels(n), QUAD, edges)


def _rmat_nzr(n, edges):
    a, b, c, d = QUAD
    return _distinct(_levels(n), (a + b, c + d), edges)


def _square_weights():
    a, b, c, d = QUAD
    return (a * a + b * c, a * b + b * d, c * a + d * c, c * b + d * d)


def _square_nnz(n, edges_a, edges_b):
    return _distinct(_levels(n), _square_weights(), _rmat_nnz(n, edges_a) * _rmat_nnz(n, edges_b))


def _square_products(n, edges_a, edges_b):
    a, b, c, d = QUAD
    return _rmat_nnz(n, edges_a) * _rmat_nnz(n, edges_b) * ((a + c) * (a + b) + (b + d) * (c + d)) ** _levels(n)


def _dcsr_bytes(nnz, nzr):
    return 4.0 * (nnz + 2 * nzr + 1)


def work(case):
    op = case["op"]
    if op in ("product", "blocks"):
        if case["pattern"] == "uniform":
            r, k, c = case["rows"], case["inner"], case["cols"]
            na, nb = case["pairs_a"], case["pairs_b"]
            products = na * nb / k
            nnz = r * c * -math.expm1(-products / (r * c))
            zr = r * -math.expm1(-na / r)
            return {"bytes": _dcsr_bytes(na, zr) + _dcsr_bytes(nb, k * -math.expm1(-nb / k)) + _dcsr_bytes(nnz, zr),
                    "flops": products}
        if case["pattern"] == "zipf":
            zr = case["n"] * case["row_share"]
            na = zr * float((_zipf_weights() * np.arange(1, ZIPF_CAP + 1)).sum())
            products = na * na / case["n"]
            return {"bytes": _dcsr_bytes(na, zr) + _dcsr_bytes(products, zr), "flops": products}
        n, m = case["n"], case["edges"]
        zr = _rmat_nzr(n, m)
        return {"bytes": _dcsr_bytes(_rmat_nnz(n, m), zr) + _dcsr_bytes(_square_nnz(n, m, m), zr),
                "flops": _square_products(n, m, m)}
    if op == "closure":
        n, sizes = case["n"], _label_sizes(case)
        total = {"bytes": 0.0, "flops": 0.0}
        for x, y, z in _rules(case):
            for k, m in ((x, sizes[x]), (y, sizes[y]), (z, sizes[z])):
                total["bytes"] += _dcsr_bytes(_rmat_nnz(n, m), _rmat_nzr(n, m))
            total["bytes"] += 4.0 * _square_nnz(n, sizes[y], sizes[z])
            total["flops"] += _square_products(n, sizes[y], sizes[z])
        return total
    if op == "kronecker":
        n, m, k = case["n"], case["edges"], case["moves"]
        nnz, zr = _rmat_nnz(n, m), _rmat_nzr(n, m)
        sr = case["states"] * -math.expm1(-k / case["states"])
        return {"bytes": _dcsr_bytes(nnz, zr) + _dcsr_bytes(k * nnz, sr * zr), "flops": k * nnz}
    if op == "union":
        n, ma, mb = case["n"], case["edges_a"], case["edges_b"]
        head = {"dcsr": lambda v, m: 2 * _rmat_nzr(n, m), "csr": lambda v, m: n, "coo": lambda v, m: v}[case["format"]]
        na, nb, nc = _rmat_nnz(n, ma), _rmat_nnz(n, mb), _rmat_nnz(n, ma + mb)
        return {"bytes": 4.0 * sum(v + head(v, m) for v, m in ((na, ma), (nb, mb), (nc, ma + mb))), "flops": na + nb}
    nnz, zr, m = _rmat_nnz(case["n"], case["edges"]), _rmat_nzr(case["n"], case["edges"]), case["edges"]
    if op == "construct":
        return {"bytes": 8.0 * m + _dcsr_bytes(nnz, zr), "flops": m}
    return {"bytes": 2 * _dcsr_bytes(nnz, zr), "flops": nnz}
