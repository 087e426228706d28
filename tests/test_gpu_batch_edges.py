"""The batched step at the edges of its tiles, every matrix against the oracle
after each of two steps: batch sizes around the workgroup's rounds, one row
that takes every triple, rows of 0 to 4,096 entries around the 32 entries met
at once, inserts before the first and after the last entry, adds, deletions to
zero and repeated coordinates; products with FP64.  Structure and update values
are compared bit for bit."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, fp64_spmv_check

pytestmark = pytest.mark.gpu


def matrix(rng, kind):
    """(rows, r, c, v): local coordinates, unique."""
    if kind == "lengths":  # rows of length 0, 1, 15 .. 65, ...
        lens = [0, 1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97, 128, 200]
        n = 256
        r = np.repeat(np.arange(len(lens)), lens)
        c = np.concatenate([np.sort(rng.permutation(n)[:k]) for k in lens])
    elif kind == "wide":  # a full row, an empty one, a long one
        n = 4096
        lens = [4096, 0, 2000, 3]
        r = np.repeat(np.arange(len(lens)), lens)
        c = np.concatenate([np.sort(rng.permutation(n)[:k]) for k in lens])
    elif kind == "one":
        return 1, np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32)
    else:
        n = int(kind)
        key = np.unique(rng.integers(0, n, 12 * n) * n + rng.integers(0, n, 12 * n))
        r, c = key // n, key % n
    v = rng.integers(1, 4, r.size).astype(np.float32) * rng.choice([-1, 1], r.size)
    return n, r.astype(np.int32), c.astype(np.int32), v.astype(np.float32)


def batch(rng, A, n, mode):
    rows = np.repeat(np.arange(A.rows), np.diff(A.off))
    br, bc = rng.integers(0, A.rows, n), rng.integers(0, A.cols, n)
    bv = rng.integers(-3, 4, n).astype(np.float32)
    if mode == "row":  # every triple in one row
        br[:] = rng.integers(0, min(A.rows, 4))
    elif A.nnz and mode == "adds":
        pick = rng.integers(0, A.nnz, n)
        br, bc, bv = rows[pick], A.col[pick], np.ones(n, np.float32) * 8
    elif A.nnz and n > 3:
        pick = rng.permutation(A.nnz)[: n // 2]
        br[: pick.size], bc[: pick.size] = rows[pick], A.col[pick]
        bv[: pick.size // 2] = -A.val[pick[: pick.size // 2]]  # deletions
        br[-n // 8:], bc[-n // 8:] = br[-n // 8], bc[-n // 8]  # repeats
    return br.astype(np.int32), bc.astype(np.int32), bv


@pytest.mark.parametrize("mode", ["mixed", "row", "adds"])
@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 2048, 4095, 4096])
def test_step_edges(mode, n):
    import torch
    import dcsr_amd
    rng = np.random.default_rng(n + len(mode))
    mats = [matrix(rng, k) for k in ("lengths", "wide", "one", "5", "300", "4096", "1000")]
    sizes = np.array([m[0] for m in mats], np.int32)
    A = [O.coo_to_csr(k, k, r, c, v) for k, r, c, v in mats]
    b = dcsr_amd.DcsrBatch(sizes, sizes, pool_factor=4.0)

    def join(parts):
        off = np.concatenate([[0], np.cumsum([p[0].size for p in parts])]).astype(np.int64)
        return (off,) + tuple(np.concatenate([p[i] for p in parts]) for i in range(3))

    b.load_coo(*join([m[1:] for m in mats]))
    x = rng.uniform(-1, 1, b.total_cols).astype(np.float32)
    for step in range(2):
        parts = [batch(rng, a, n, mode) for a in A]
        if step:
            parts[4] = tuple(np.resize(p, 4097) for p in parts[4])  # one matrix over the limit: untouched
        y = b.step(*join(parts), x=torch.from_numpy(x).cuda())
        code, per = b.status()
        assert code == (8 if step else 0) and [i for i in range(7) if per[i]] == ([4] if step else [])
        A = [a if step and i == 4 else O.update(a, *p) for i, (a, p) in enumerate(zip(A, parts))]
        off, col, val = (t.cpu().numpy() for t in b.to_csr())
        for i, a in enumerate(A):
            r0, r1, c0 = int(b.row_base[i]), int(b.row_base[i + 1]), int(b.col_base[i])
            got = O.Csr(a.rows, a.cols, off[r0:r1 + 1] - off[r0], col[off[r0]:off[r1]], val[off[r0]:off[r1]])
            assert_same_structure(got, a)
            fp64_spmv_check(a, x[c0:c0 + a.cols], y.cpu().numpy()[r0:r1])
    b.close()
