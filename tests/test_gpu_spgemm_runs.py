"""SpGEMM rows of the workgroup classes with few columns: as many runs of equal
columns as partials allow on both sides of the line past which their starts are
listed (one in four keys of a step), runs of uneven length, and rows that start
crowded and go on with more starts than the list holds, or the other way round.  Sums follow the host path's order: compared bit for bit."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure

pytestmark = pytest.mark.gpu


def product(rows, cols):
    """rows: the columns of one row of the product in generation order (ascending
    stretches, each a row of B)."""
    import dcsr_amd
    from tests.helpers import to_host_csr
    rng = np.random.default_rng(len(rows))
    br, bc, ar, ac, n = [], [], [], [], 0
    for i, g in enumerate(rows):
        cut = np.flatnonzero(np.concatenate([[True], g[1:] <= g[:-1]]))
        piece = np.repeat(np.arange(cut.size), np.diff(np.concatenate([cut, [g.size]])))
        br.append(n + piece)
        bc.append(g)
        ar.append(np.full(cut.size, i))
        ac.append(n + np.arange(cut.size))
        n += cut.size
    br, bc, ar, ac = (np.concatenate(x).astype(np.int32) for x in (br, bc, ar, ac))
    B = O.coo_to_csr(n, cols, br, bc, rng.uniform(-1, 1, br.size).astype(np.float32))
    A = O.coo_to_csr(len(rows), n, ar, ac, rng.uniform(-1, 1, ar.size).astype(np.float32))
    mA, mB = dcsr_amd.DcsrMatrix(A.rows, A.cols), dcsr_amd.DcsrMatrix(B.rows, B.cols)
    mA.load_csr(A.off, A.col, A.val)
    mB.load_csr(B.off, B.col, B.val)
    mC = dcsr_amd.spgemm(mA, mB)
    assert_same_structure(to_host_csr(mC), O.spgemm(A, B), values="exact")
    for m in (mA, mB, mC):
        m.close()


@pytest.mark.parametrize("cols", [200_000, 1 << 26])
@pytest.mark.parametrize("P", [1025, 4095, 4096, 4097, 8192, 8193, 16383, 16384])
def test_few_columns(P, cols):
    rng = np.random.default_rng(P)
    rows = []
    for D in (1, 2, 63, P // 9, P // 4 - 1, P // 4, P // 4 + 1, P // 3, P // 2):
        g = np.arange(P) % D  # every column P / D times
        rows.append(g * (cols // D))
    # uneven: half of the partials in one column, one in another
    u = np.sort(rng.choice(cols, 40, replace=False))
    parts = [u[rng.random(u.size) < 0.3] for _ in range(P // 12)]
    h = np.concatenate([np.union1d(p, u[7]) for p in parts])
    rows.append(np.concatenate([h, np.full(P, u[7])])[:P])
    product(rows, cols)


@pytest.mark.parametrize("P,NT", [(4096, 256), (16384, 1024), (5000, 1024), (1300, 256)])
@pytest.mark.parametrize("lead", [0, 1, 1000])
def test_from_few_columns_to_many(P, NT, lead):
    # `lead` columns of one partial, one of NT, then of one partial each; and reversed
    rest = max(P - lead - NT, 0)
    rows = []
    for tail in (0, 1):
        runs = np.concatenate([np.ones(lead, int), [P - lead - rest], np.ones(rest, int)])
        if tail:
            runs = runs[::-1]
        k = np.repeat(np.arange(runs.size), runs)
        first = np.concatenate([[True], k[1:] != k[:-1]])
        rows.append(np.concatenate([k[first], k[~first]]))
    product(rows, P)
