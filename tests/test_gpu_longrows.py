"""Tiles of many short rows and one long one: the row's chain of additions at
its remainders, and the two ways SpMV 2 forms q on either side of the length
at which a row is no longer walked by one thread."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from hbicg import Plan, make_params
from hbicg import problems as P

pytestmark = pytest.mark.gpu


def _matrix(n, at, length, seed):
    """n rows of three entries; row `at` has `length` (all distinct columns, its diagonal among them)."""
    ptr, cols = [0], []
    for i in range(n):
        if i == at:
            c = (i + np.arange(length) * (n // length)) % n
        else:
            c = np.array([i, (i + 7) % n, (i + n // 2) % n])
        cols.append(np.unique(c))
        ptr.append(ptr[-1] + len(cols[-1]))
    col = np.concatenate(cols)
    val = P.uniform(seed, 3, len(col), -1.0, 1.0)
    row = np.repeat(np.arange(n), np.diff(ptr))
    val[row == col] = 2.0 + np.bincount(row, weights=np.abs(val), minlength=n)[row[row == col]]
    return P.CSR(np.array(ptr, np.uint32), col.astype(np.uint32), val, n)


@pytest.mark.parametrize("n", [250, 1100])      # all rows, and 256 of them, in the long row's tile
@pytest.mark.parametrize("length", [31, 32, 33, 39, 40, 41, 47, 48, 55, 56, 63, 64, 65, 200, 243])
def test_long_row(n, length):
    A = _matrix(n, n // 3, length, 4)
    b = torch.as_tensor(P.uniform(2, 1, n, -1.0, 1.0)).cuda()
    out = []
    for q_mode in (1, 2):
        pl = Plan(A, 3, make_params(tol=1e-10, graph=0, q_mode=q_mode))
        x = torch.zeros((3, n), dtype=torch.float64, device="cuda")
        k, _, rep = pl.solve(b, P.logspace_shifts(3, 1e-3, 1.0), 0, x)
        y = pl.spmv(b)
        pl.close()
        out.append((k, x, y))
    assert out[0][0] == out[1][0] and torch.equal(out[0][1], out[1][1])
    # a sum of m products: at most m roundings of the sum of their sizes
    row = np.repeat(np.arange(n), np.diff(A.ptr.astype(np.int64)))
    prod = A.val * b.cpu().numpy()[A.col]
    want, size = np.bincount(row, weights=prod, minlength=n), np.bincount(row, weights=np.abs(prod), minlength=n)
    m = np.diff(A.ptr.astype(np.int64)) + 1
    assert np.all(np.abs(out[0][2].cpu().numpy() - want) <= 2 * m * 2.0 ** -53 * size)
