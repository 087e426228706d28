"""Timed cases of the Dynamic-CSR engine: what a program that keeps a sparse
matrix on the GPU has it do, from one 1,000-triple update of a 256-row matrix
to a product of 2M-row matrices.

Kinds (each through the public classes of ``dcsr_amd``):

* ``stream``  -- a sliding window over a graph: one batch of triples enters
  (insert-or-add, some of it deletions), a product is taken, the matrix is
  saved as CSR; then the batch leaves again (the same triples negated, so new
  coordinates cancel to zero and are removed) and a product follows.  A pass
  leaves the structure it found, so it can be repeated.
* ``product`` -- y = A x, or Y = A X with k columns, of a resident matrix.
* ``square``  -- C = A A, and C as CSR.
* ``batch``   -- many small matrices stepped together: every matrix takes its
  own triples and multiplies, all are saved, then the triples leave again.
* ``ingest``  -- a matrix read into an existing handle (unordered triples with
  a few repeated coordinates, or CSR), one product, and out again as CSR.
* ``serve``   -- a burst of queries and updates at the request loop.

Saved matrices go into CSR buffers that the program keeps, of a capacity that
bounds every matrix of the case (entries past the matrix's own stay zero).

Values are in (0, 1] as edge weights are; the matrices are the banded, Zipf
(web graph) and Poisson patterns of ``dcsr_amd.workloads``, drawn on the GPU.
"""
from __future__ import annotations

import ctypes
import math

import torch

import dcsr_amd

DEV = "cuda"


def listed():
    return [
        # the reference drivers' own flow on its bundled 256-row matrix: the
        # smallest call, all launches and latency; every update reports back
        dict(name="stream_banded_256", kind="stream", graph="banded", rows=256, nnz=3_000, batch=1_000,
             dels=0.0, sync=True, pool=2.0),
        # a small graph fed by asynchronous batches, odd sizes
        dict(name="stream_20k", kind="stream", graph="powerlaw", rows=20_011, nnz=200_003, batch=5_001,
             dels=0.1, sync=False, pool=8.0),
        # a large graph that takes small batches, deletions among them, as a
        # live service feeds it
        dict(name="stream_1m_10k", kind="stream", graph="powerlaw", rows=1_000_003, nnz=16_000_000, batch=10_000,
             dels=0.3, sync=False, pool=4.0),
        # the benchmark's headline: web graph, 1M-triple asynchronous batches
        dict(name="stream_325k_1m", kind="stream", graph="powerlaw", rows=325_557, nnz=3_200_000, batch=1_000_000,
             dels=0.0, sync=False, pool=64.0),
        # the largest update: a 2M-row matrix takes 4M triples in one call
        dict(name="stream_2m_4m", kind="stream", graph="poisson", rows=2_000_000, nnz=16_000_000, batch=4_000_000,
             dels=0.1, sync=True, pool=4.0),
        # products of resident matrices: HBM-sized, and with 16 columns
        dict(name="spmv_10m", kind="product", graph="powerlaw", rows=10_000_000, nnz=160_000_000, k=1, pool=1.0),
        dict(name="spmm_1m_k16", kind="product", graph="powerlaw", rows=1_000_003, nnz=16_000_000, k=16, pool=1.0),
        # sparse products: short even rows, and a graph with hub rows
        dict(name="square_2m", kind="square", graph="poisson", rows=2_000_000, nnz=16_000_000, pool=2.0),
        dict(name="square_graph_100k", kind="square", graph="powerlaw", rows=100_003, nnz=1_000_000, pool=2.0),
        # 4,096 small matrices x 2,000 triples per step, one graph launch each
        dict(name="batch_4096", kind="batch", count=4_096, low=64, high=4_096, mean=16.0, per=2_000, graph=True),
        # an unordered edge list becomes a matrix
        dict(name="ingest_3m", kind="ingest", graph="powerlaw", rows=325_557, nnz=3_200_000, form="coo", pool=2.0),
        # 36 queries of 1 to 32 columns and 4 updates arrive at once
        dict(name="serve_1m", kind="serve", graph="powerlaw", rows=1_000_003, nnz=16_000_000, queries=36, updates=4,
             low=1_000, high=100_000, max_cols=64),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["stream"] * 5 + ["product"] * 2 + ["square"] * 2 + ["batch", "ingest", "ingest", "serve"])
    graph = rng.choice(["powerlaw", "powerlaw", "poisson"])
    if kind == "stream":
        rows = _log(rng, 256, 2_000_000)
        nnz = rows * rng.randint(5, 16)
        return dict(kind=kind, graph=graph, rows=rows, nnz=nnz, batch=_log(rng, 500, min(4_000_000, nnz // 2)),
                    dels=rng.choice([0.0, 0.1, 0.3]), sync=rng.random() < 0.4, pool=rng.choice([2.0, 4.0, 8.0, 64.0]))
    if kind == "product":
        rows = _log(rng, 2_000, 8_000_000)
        k = rng.choice([1, 1, 1, 2, 3, 4, 7, 8, 16, 17, 32])
        nnz = min(rows * rng.randint(4, 20), 120_000_000 // max(1, k // 4))
        return dict(kind=kind, graph=graph, rows=rows, nnz=max(nnz, rows), k=k, pool=1.0)
    if kind == "square":
        rows = _log(rng, 256, 1_500_000)
        mean = rng.randint(3, 8) if graph == "poisson" else rng.randint(3, 6)
        return dict(kind=kind, graph=graph, rows=rows, nnz=rows * mean, pool=2.0)
    if kind == "batch":
        high = _log(rng, 200, 4_096)
        return dict(kind=kind, count=_log(rng, 8, 3_000), low=64, high=high, mean=float(rng.randint(4, 16)),
                    per=_log(rng, 100, 3_000), graph=rng.random() < 0.6)
    if kind == "ingest":
        rows = _log(rng, 300, 2_000_000)
        return dict(kind=kind, graph=graph, rows=rows, nnz=rows * rng.randint(4, 12), form=rng.choice(["coo", "csr"]),
                    pool=2.0)
    rows = _log(rng, 20_000, 1_000_000)
    return dict(kind=kind, graph=graph, rows=rows, nnz=rows * rng.randint(6, 14), queries=rng.randint(12, 36),
                updates=2 * rng.randint(1, 2), low=1_000, high=100_000, max_cols=64)


# --------------------------------------------------------------------------
# inputs, drawn on the GPU from the seed alone
# --------------------------------------------------------------------------

def _weights(n, gen):
    return 1.0 - torch.rand(n, generator=gen, device=DEV)


def _triples(case, gen):
    """Sorted unique coordinates (int64 rows, cols) and float32 weights."""
    R, nnz = case["rows"], case["nnz"]
    if case["graph"] == "banded":
        i = torch.arange(R, device=DEV)
        d = torch.arange(1, min(41, R), device=DEV)
        rr, dd = i.repeat_interleave(d.numel()), d.repeat(R)
        keep = (rr + dd < R) & (torch.rand(rr.numel(), generator=gen, device=DEV) < 0.1457)
        rr, cc = rr[keep], rr[keep] + dd[keep]
        key = torch.cat([i * R + i, rr * R + cc, cc * R + rr])
    else:
        mean = nnz / R
        if case["graph"] == "poisson":
            deg = torch.poisson(torch.full((R,), mean, device=DEV), generator=gen).to(torch.int64)
        else:
            # Zipf(2.1) out-degrees scaled to the mean, capped at R / 120
            cap = float(max(R // 120, 64))
            z = torch.floor((1.0 - torch.rand(R, generator=gen, device=DEV, dtype=torch.float64)) ** (-1.0 / 1.1))
            lo, hi = 1e-3, 1e3
            for _ in range(40):
                mid = 0.5 * (lo + hi)
                small = float(torch.clamp(torch.ceil(mid * z), 1.0, cap).sum()) < nnz
                lo, hi = (mid, hi) if small else (lo, mid)
            deg = torch.clamp(torch.ceil(lo * z), 1.0, cap).to(torch.int64)
        deg = torch.clamp(deg, max=R)
        rr = torch.repeat_interleave(torch.arange(R, device=DEV), deg)
        key = rr * R + torch.randint(0, R, (rr.numel(),), generator=gen, device=DEV)
    key = torch.unique(key)
    return key // R, key % R, _weights(key.numel(), gen)


def _change(r, c, v, ncols, n, dels, gen):
    """One batch in random order: `dels` of it removes stored entries, as many
    of the rest add to stored entries as bring new columns to rows drawn by
    degree.  Its negation takes it back."""
    nnz = r.numel()
    nd = int(n * dels)
    na = (n - nd) // 2
    half = max(nnz // 2, 1)  # removals come from one half of the entries, additions from the other
    gone = 2 * torch.unique(torch.randint(0, half, (nd,), generator=gen, device=DEV)) if nd else \
        torch.zeros(0, dtype=torch.int64, device=DEV)
    add = 2 * torch.randint(0, max((nnz - 1) // 2, 1), (na,), generator=gen, device=DEV) + (1 if nnz > 1 else 0)
    m = n - gone.numel() - na
    at = torch.randint(0, nnz, (m,), generator=gen, device=DEV)
    rows = torch.cat([r[gone], r[add], r[at]])
    cols = torch.cat([c[gone], c[add], torch.randint(0, ncols, (m,), generator=gen, device=DEV)])
    vals = torch.cat([-v[gone], _weights(na + m, gen)])
    p = torch.randperm(n, generator=gen, device=DEV)
    return rows[p].to(torch.int32), cols[p].to(torch.int32), vals[p]


def _sizes(case):
    """Rows of the small matrices, evenly spread over their logarithm."""
    lo, hi = math.log(case["low"]), math.log(case["high"])
    u = (torch.arange(case["count"], device=DEV, dtype=torch.float64) + 0.5) / case["count"]
    return torch.exp(lo + (hi - lo) * u).round().to(torch.int64)


def _room(case):
    """Entries that no matrix of the case exceeds."""
    kind = case["kind"]
    if kind == "batch":
        N = int(_sizes(case).sum()) * (case["mean"] + 1)
        return int(N + 8 * math.sqrt(N) + 64) + case["count"] * case["per"]
    R, N = case["rows"], case["nnz"]
    if kind == "square":
        return min(R * R, int(N * N / R * (1 + 64 / math.sqrt(R))) + 4_096)
    return int(N + 8 * math.sqrt(N) + 64) + case.get("batch", 0)


def _many(case, gen):
    """Sizes of the small matrices, their triples with local coordinates in
    matrix order, and one batch for each, as many triples each."""
    n, per = case["count"], case["per"]
    size = _sizes(case)[torch.randperm(n, generator=gen, device=DEV)]
    base = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    base[1:] = torch.cumsum(size, 0)
    R = int(base[-1])
    deg = torch.poisson(torch.full((R,), case["mean"], device=DEV), generator=gen).to(torch.int64) + 1
    row = torch.repeat_interleave(torch.arange(R, device=DEV), deg)
    mat = torch.bucketize(row, base[1:], right=True)

    def column(m):
        return (torch.rand(m.numel(), generator=gen, device=DEV, dtype=torch.float64) * size[m]).to(torch.int64)

    key = torch.unique(row * 4_096 + column(mat))
    row, col = key // 4_096, key % 4_096
    mat = torch.bucketize(row, base[1:], right=True)
    val = _weights(key.numel(), gen)
    off = torch.searchsorted(mat, torch.arange(n + 1, device=DEV))
    # the batch: half adds to stored entries of the matrix, half new columns
    bm = torch.arange(n, device=DEV).repeat_interleave(per)
    span = (off[1:] - off[:-1])[bm]
    pick = off[bm] + (torch.rand(bm.numel(), generator=gen, device=DEV, dtype=torch.float64) * span).to(torch.int64)
    brow = row[pick]
    old = torch.rand(bm.numel(), generator=gen, device=DEV) < 0.5
    bcol = torch.where(old, col[pick], column(bm))
    boff = torch.arange(n + 1, device=DEV) * per
    return size, base, (off, row, col, val), (boff, brow, bcol, _weights(bm.numel(), gen))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _i32(t):
    return t.to(torch.int32)


def _offsets(r, rows):
    return _i32(torch.searchsorted(r, torch.arange(rows + 1, device=DEV)))


def _inputs(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "batch":
        size, base, mats, batch = _many(case, gen)
        return dict(size=size, base=base, mats=mats, batch=batch, x=_weights(int(base[-1]), gen))
    R = case["rows"]
    r, c, v = _triples(case, gen)
    d = dict(r=r, c=c, v=v)
    if kind == "stream":
        d["batch"] = _change(r, c, v, R, case["batch"], case["dels"], gen)
        d["x"] = _weights(R, gen)
    elif kind == "product":
        k = case["k"]
        d["x"] = _weights(R * k, gen).reshape(R, k) if k > 1 else _weights(R, gen)
    elif kind == "ingest":
        if case["form"] == "coo":
            twice = torch.randint(0, r.numel(), (r.numel() // 100,), generator=gen, device=DEV)
            d["r"], d["c"] = torch.cat([r, r[twice]]), torch.cat([c, c[twice]])
            d["v"] = torch.cat([v, _weights(twice.numel(), gen)])
            p = torch.randperm(d["r"].numel(), generator=gen, device=DEV)
            d["r"], d["c"], d["v"] = d["r"][p], d["c"][p], d["v"][p]
        d["x"] = _weights(R, gen)
    elif kind == "serve":
        # widths of the mix 55 / 20 / 15 / 10 %, in a fixed scattered order
        mix = [1] * 11 + [4] * 4 + [16] * 3 + [32] * 2
        ks = [mix[7 * i % 20] for i in range(case["queries"])]
        d["X"] = {k: _weights(R * k, gen).reshape(R, k) for k in (1, 4, 16, 32)}
        ups = []
        for j in range(case["updates"] // 2):
            u = (j + 0.5) / (case["updates"] // 2)
            n = int(math.exp(math.log(case["low"]) + u * (math.log(case["high"]) - math.log(case["low"]))))
            ups.append(_change(r, c, v, R, n, 0.0, gen))
        # updates enter in the first half of the requests and leave in the second
        reqs, half = [("query", k) for k in ks], case["queries"] // 2
        for j, _ in enumerate(ups):
            reqs.insert((j + 1) * half // (len(ups) + 1) + j, ("in", j))
        back = len(reqs) - (case["queries"] - half)
        for j, _ in enumerate(ups):
            reqs.insert(back + (j + 1) * half // (len(ups) + 1) + j, ("out", j))
        d["ups"], d["reqs"] = ups, reqs
    return d


# --------------------------------------------------------------------------
# what a program holds before the call, and the call
# --------------------------------------------------------------------------

def _buffers(case, rows):
    n = _room(case)
    return (torch.zeros(rows + 1, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV),
            torch.zeros(n, device=DEV))


def _save(handle, csr, flags=0):
    """The matrix of a handle into the program's own CSR buffers."""
    n = ctypes.c_int64(0)
    dcsr_amd.check(dcsr_amd.lib().dcsr_export_csr(
        handle, csr[0].data_ptr(), csr[1].data_ptr(), csr[2].data_ptr(), csr[1].numel(), ctypes.byref(n), flags,
        torch.cuda.current_stream().cuda_stream), "dcsr_export_csr")
    return csr


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "batch":
        size = d["size"].cpu().numpy()
        b = dcsr_amd.DcsrBatch(size, size, pool_factor=8.0)
        base, (off, row, col, val) = d["base"], d["mats"]
        which = torch.bucketize(row, base[1:], right=True)
        b.load_coo(off, _i32(row - base[which]), _i32(col), val)
        boff, brow, bcol, bval = d["batch"]
        bm = torch.arange(case["count"], device=DEV).repeat_interleave(case["per"])
        s.update(b=b, off=boff, r=_i32(brow - base[bm]), c=_i32(bcol), v=bval, back=-bval, x=d["x"],
                 y=torch.empty(b.total_rows, device=DEV), y1=torch.empty(b.total_rows, device=DEV))
        s["v_in"] = torch.empty_like(bval)  # the step's own input buffer, refilled before each step
        s["csr"] = _buffers(case, b.total_rows)
        return s
    R = case["rows"]
    if kind == "ingest":
        s["m"] = dcsr_amd.DcsrMatrix(R, R, pool_factor=case["pool"])
        if case["form"] == "csr":
            s.update(off=_offsets(d["r"], R), c=_i32(d["c"]), v=d["v"])
        else:
            s.update(r=_i32(d["r"]), c=_i32(d["c"]), v=d["v"])
        s.update(x=d["x"], y=torch.empty(R, device=DEV), csr=_buffers(case, R))
        return s
    m = dcsr_amd.DcsrMatrix(R, R, pool_factor=case.get("pool", 8.0))
    m.load_csr(_offsets(d["r"], R), _i32(d["c"]), d["v"])
    s["m"] = m
    if kind == "stream":
        r, c, v = d["batch"]
        s.update(r=r, c=c, v=v, back=-v, x=d["x"], y=torch.empty(R, device=DEV), y2=torch.empty(R, device=DEV),
                 csr=_buffers(case, R))
    elif kind == "product":
        s.update(x=d["x"], y=torch.empty_like(d["x"]))
    elif kind == "square":
        s.update(out=dcsr_amd.DcsrMatrix(R, R), csr=_buffers(case, R))
    elif kind == "serve":
        reqs = []
        for what, j in d["reqs"]:
            if what == "query":
                reqs.append((d["X"][j], torch.empty((R, j), device=DEV)))
            else:
                r, c, v = d["ups"][j]
                reqs.append((r, c, v if what == "in" else -v))
        s.update(server=dcsr_amd.DcsrServer(m, max_cols=case["max_cols"]), reqs=reqs)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "stream":
        m, flags = state["m"], 0 if case["sync"] else dcsr_amd.UPDATE_NOSYNC
        m.UpdateMatrix(state["r"], state["c"], state["v"], flags=flags)
        m.spmv(state["x"], state["y"])
        saved = _save(m.handle, state["csr"])
        m.UpdateMatrix(state["r"], state["c"], state["back"], flags=flags)
        m.spmv(state["x"], state["y2"])
        return dict(csr=saved, y=state["y"], after=state["y2"])
    if kind == "product":
        m = state["m"]
        return m.spmv(state["x"], state["y"]) if case["k"] == 1 else m.spmm(state["x"], state["y"])
    if kind == "square":
        return _save(dcsr_amd.spgemm(state["m"], state["m"], state["out"]).handle, state["csr"])
    if kind == "batch":
        b, graph = state["b"], case["graph"]
        state["v_in"].copy_(state["v"])
        b.step(state["off"], state["r"], state["c"], state["v_in"], x=state["x"], y=state["y"], graph=graph)
        saved = _save(dcsr_amd.lib().dcsr_batch_handle(b._b), state["csr"])
        state["y1"].copy_(state["y"])
        state["v_in"].copy_(state["back"])
        b.step(state["off"], state["r"], state["c"], state["v_in"], x=state["x"], y=state["y"], graph=graph)
        return dict(csr=saved, y=state["y1"], after=state["y"])
    if kind == "ingest":
        m = state["m"]
        if case["form"] == "coo":
            m.LoadMatrix(state["r"], state["c"], state["v"])
        else:
            m.load_csr(state["off"], state["c"], state["v"])
        m.spmv(state["x"], state["y"])
        return dict(csr=_save(m.handle, state["csr"], dcsr_amd.EXPORT_CANONICAL), y=state["y"])
    srv = state["server"]
    for q in state["reqs"]:
        if len(q) == 3:
            srv.update(*q)
        elif q[0].shape[1] == 1:
            srv.spmv(q[0][:, 0], q[1][:, 0])
        else:
            srv.spmm(*q)
    srv.drain()
    return [q[1] for q in state["reqs"] if len(q) == 2]


# --------------------------------------------------------------------------
# what a pass cannot do without, and its results in 64 bits
# --------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "batch":
        R = case["count"] * (case["high"] - case["low"]) / math.log(case["high"] / case["low"])
        N, n = R * (case["mean"] + 1), case["count"] * case["per"]
        step = 12 * n + 8 * n + 8 * min(R, n) + 8 * N + 12 * R
        return dict(bytes=2 * step + 16 * N + 4 * R, flops=4 * N + 2 * n)
    R, N = case["rows"], case["nnz"]
    mul = 4 * (R + 1) + 8 * N + 8 * R  # A, x and y once each
    if kind == "stream":
        n = case["batch"]
        change = 12 * n + 8 * n + 8 * min(R, n)  # triples in, entries out, touched rows' table
        return dict(bytes=2 * change + 2 * mul + 16 * N + 4 * R, flops=4 * N + 2 * n)
    if kind == "product":
        k = case["k"]
        return dict(bytes=4 * (R + 1) + 8 * N + 8 * k * R, flops=2 * k * N)
    if kind == "square":
        # partial products of uniform columns: N times the mean row, gathered
        # once from B and stored once in C
        P = N * N / R
        return dict(bytes=16 * N + 8 * P + 12 * R, flops=2 * P)
    if kind == "ingest":
        return dict(bytes=12 * N + 8 * N + 8 * R + mul + 8 * N + 4 * R, flops=2 * N)
    # each stretch of queries between two updates reads A once
    cols = case["queries"] * (.55 + .2 * 4 + .15 * 16 + .1 * 32)
    return dict(bytes=(case["updates"] + 1) * 8 * N + 8 * cols * R, flops=2 * cols * N)


def _csr64(rows, key, val, R, C):
    key, inv = torch.unique(key, return_inverse=True)
    s = torch.zeros(key.numel(), dtype=torch.float64, device=DEV).index_add_(0, inv, val)
    keep = s != 0
    return key[keep] // C, key[keep] % C, s[keep]


def _times(r, c, v, x, R):
    y = torch.zeros(R, dtype=torch.float64, device=DEV)
    step = 1 << 25
    for i in range(0, r.numel(), step):
        y.index_add_(0, r[i:i + step], v[i:i + step].double() * x[c[i:i + step]].double())
    return y


def _padded(v, case):
    out = torch.zeros(_room(case), dtype=torch.float64, device=DEV)
    out[:v.numel()] = v
    return out


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "batch":
        base, (_, row, col, val), (_, brow, bcol, bval) = d["base"], d["mats"], d["batch"]
        R = int(base[-1])
        start = base[torch.bucketize(torch.arange(R, device=DEV), base[1:], right=True)]
        after = _times(row, start[row] + col, val, d["x"], R)
        r, c, v = _csr64(R, torch.cat([row, brow]) * 4_096 + torch.cat([col, bcol]),
                         torch.cat([val, bval]).double(), R, 4_096)
        return dict(csr=(None, None, _padded(v, case)), y=_times(r, start[r] + c, v, d["x"], R), after=after)
    R = case["rows"]
    r, c, v = d["r"], d["c"], d["v"]
    if kind == "stream":
        br, bc, bv = (t.to(torch.int64) if t.dtype == torch.int32 else t for t in d["batch"])
        nr, nc, nv = _csr64(R, torch.cat([r, br]) * R + torch.cat([c, bc]), torch.cat([v, bv]).double(), R, R)
        return dict(csr=(None, None, _padded(nv, case)), y=_times(nr, nc, nv, d["x"], R), after=_times(r, c, v, d["x"], R))
    if kind == "product":
        if case["k"] == 1:
            return _times(r, c, v, d["x"], R)
        return torch.stack([_times(r, c, v, d["x"][:, j], R) for j in range(case["k"])], 1)
    if kind == "square":
        off = torch.searchsorted(r, torch.arange(R + 1, device=DEV))
        n = (off[1:] - off[:-1])[c]  # partial products of each entry
        total = int(n.sum())
        which = torch.repeat_interleave(torch.arange(r.numel(), device=DEV), n)
        first = torch.cumsum(n, 0) - n
        b = off[c][which] + torch.arange(total, device=DEV) - first[which]
        val = v[which].double() * v[b].double()
        key = r[which] * R + c[b]
        del which, b
        return (None, None, _padded(_csr64(R, key, val, R, R)[2], case))
    if kind == "ingest":
        y = _times(r, c, v, d["x"], R)
        return dict(csr=(None, None, _padded(_csr64(R, r * R + c, v.double(), R, R)[2], case)), y=y)
    # requests: the matrix of a query is the first one plus the batches that are in
    outs, inside = [], []
    kept = {}
    for what, j in d["reqs"]:
        if what == "in":
            inside.append(j)
        elif what == "out":
            inside.remove(j)
        else:
            X = d["X"][j]
            if j not in kept:
                kept[j] = torch.stack([_times(r, c, v, X[:, i], R) for i in range(j)], 1)
            Y = kept[j].clone()
            for u in inside:
                br, bc, bv = d["ups"][u]
                Y += torch.stack([_times(br.to(torch.int64), bc.to(torch.int64), bv, X[:, i], R) for i in range(j)], 1)
            outs.append(Y)
    return outs
