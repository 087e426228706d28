"""The batched step where rows take many triples: 63 to 66 of them in one row (the
rank inside a row gives way to a sort of the whole batch past 64), every triple
in one row or at one coordinate, full and ragged batches.  Sums run in arrival
order: structure and values are compared with the oracle's bit for bit, products
with FP64."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, fp64_spmv_check

pytestmark = pytest.mark.gpu


def triples(rng, n, size, mode):
    if mode == "row":
        r, c = np.full(n, size // 3), rng.integers(0, size, n)
    elif mode == "coordinate":
        r, c = np.full(n, size - 1), np.full(n, size // 2)
    elif mode == "few":
        r, c = rng.integers(0, 4, n) * (size // 5), rng.integers(0, 4, n)
    else:  # rows of `mode` triples each
        r, c = np.arange(n) // mode % size, rng.integers(0, size, n)
    p = rng.permutation(n)
    return r[p].astype(np.int32), c[p].astype(np.int32), rng.uniform(-1, 1, n).astype(np.float32)


@pytest.mark.parametrize("mode", ["row", "coordinate", "few", 63, 64, 65, 66])
@pytest.mark.parametrize("n", [64, 65, 1_000, 4_095, 4_096])
def test_crowded_rows(mode, n):
    import torch
    import dcsr_amd
    rng = np.random.default_rng(n)
    sizes = np.array([4_096, 300, 70, 1_000], np.int32)
    b = dcsr_amd.DcsrBatch(sizes, sizes, pool_factor=8.0, min_pool=1 << 18)
    A = []
    for k in sizes:
        r, c = rng.integers(0, k, 5 * k).astype(np.int32), rng.integers(0, k, 5 * k).astype(np.int32)
        key = np.unique(r.astype(np.int64) * k + c)
        A.append(O.coo_to_csr(k, k, (key // k).astype(np.int32), (key % k).astype(np.int32),
                              rng.uniform(0, 1, key.size).astype(np.float32)))

    def join(parts):
        off = np.concatenate([[0], np.cumsum([p[0].size for p in parts])]).astype(np.int64)
        return (off,) + tuple(np.concatenate([p[i] for p in parts]) for i in range(3))

    b.load_coo(*join([(np.repeat(np.arange(a.rows), np.diff(a.off)).astype(np.int32), a.col, a.val) for a in A]))
    x = rng.uniform(-1, 1, b.total_cols).astype(np.float32)
    for _ in range(2):
        parts = [triples(rng, n, int(k), mode) for k in sizes]
        y = b.step(*join(parts), x=torch.from_numpy(x).cuda())
        assert b.status()[0] == 0
        A = [O.update(a, *p) for a, p in zip(A, parts)]
        off, col, val = (t.cpu().numpy() for t in b.to_csr())
        for i, a in enumerate(A):
            r0, r1, c0 = int(b.row_base[i]), int(b.row_base[i + 1]), int(b.col_base[i])
            got = O.Csr(a.rows, a.cols, off[r0:r1 + 1] - off[r0], col[off[r0]:off[r1]], val[off[r0]:off[r1]])
            assert_same_structure(got, a)
            fp64_spmv_check(a, x[c0:c0 + a.cols], y.cpu().numpy()[r0:r1])
    b.close()
