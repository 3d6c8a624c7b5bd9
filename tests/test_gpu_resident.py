"""The resident form of the default order (many iterations per launch) against
the launch-per-phase kernels: bitwise the same, at the sizes where its tiles,
columns of partial sums and row ownership change, for every matrix form, with
seed switches, windows closed by the growth guard, and the hand-over to
launches."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from hbicg import Batch, Plan, make_params
from hbicg import problems as P

pytestmark = pytest.mark.gpu


def _banded(n, diags, seed, values):
    """A diagonally dominant matrix on the given diagonals; values: "const"
    (one per diagonal) or "full" (one per entry).  Every fifth row lacks the
    entries on odd diagonals."""
    rows, cols, vals = [], [], []
    i = np.arange(n)
    for t, o in enumerate(diags):
        ok = (i + o >= 0) & (i + o < n)
        if t % 2 and o:
            ok &= i % 5 != 0
        c = (8.0 if o == 0 else -0.4 - 0.05 * t)
        v = np.full(n, c) if values == "const" else c * P.uniform(seed, 10 + t, n, 0.5, 1.5)
        rows.append(i[ok]); cols.append((i + o)[ok]); vals.append(v[ok])
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    at = np.lexsort((c, r))
    ptr = np.zeros(n + 1, np.uint32)
    ptr[1:] = np.cumsum(np.bincount(r, minlength=n))
    return P.CSR(ptr, c[at].astype(np.uint32), v[at], n)


def _run(A, M, seed, lo=1e-3, b_seed=1, **kw):
    """(k, x, r, stop iterations, switches, trace) of one solve."""
    dev = "cuda"
    b = torch.as_tensor(P.uniform(b_seed, 1, A.n, -1.0, 1.0)).to(dev)
    pl = Plan(A, M, make_params(tol=1e-10, graph=1, **kw))
    x, r = torch.zeros((M, A.n), dtype=torch.float64, device=dev), torch.empty_like(b)
    out = []
    for _ in range(2):   # a plan's second solve starts from what the first left
        x.zero_()
        k, _, rep = pl.solve(b, P.logspace_shifts(M, lo, 1.0), seed, x, r)
        _, stop, sw = pl.report()
        out.append((k, x.clone(), r.clone(), stop.copy(), list(sw), rep["status"],
                    pl.residual_trace() if kw.get("trace") else None))
    pl.close()
    return out


def _same(got, want):
    for g, w in zip(got, want):
        assert g[0] == w[0] and g[4] == w[4] and g[5] == w[5]
        assert np.array_equal(g[3], w[3])
        for a, c in ((g[1], w[1]), (g[2], w[2])):   # a NaN (one row solved exactly breaks down) equals a NaN
            assert torch.allclose(a, c, rtol=0.0, atol=0.0, equal_nan=True)
        if w[6] is not None:
            assert np.array_equal(g[6], w[6], equal_nan=True)


# n: one row, tails of 1, 128 and 129 rows (lanes per row of the last tile),
# one workgroup's last size and the next (16 / 17 tiles), a full column set
# (256 tiles), two and four tiles a column, the slot counts 2 (1024 tiles up)
SIZES = [1, 2, 255, 256, 257, 4 * 256, 4 * 256 + 128, 8 * 256 + 129, 16 * 256, 16 * 256 + 1, 20 * 256 + 64,
         255 * 256 + 3, 256 * 256, 256 * 256 + 1, 512 * 256, 512 * 256 + 130, 1024 * 256, 1024 * 256 + 17]


@pytest.mark.parametrize("values", ["const", "full"])
@pytest.mark.parametrize("n", SIZES)
def test_sizes(n, values):
    A = _banded(n, [-37, -1, 0, 1, 37], 3, values)
    kw = dict(value_index=values == "const")
    _same(_run(A, 5, 2, **kw), _run(A, 5, 2, fused=0, **kw))


# more than 2048 tiles: the seed update's partial sums chain tiles 2048 apart
@pytest.mark.parametrize("n", [2048 * 256, 2048 * 256 + 5, 4096 * 256 - 100, 4096 * 256 + 1, 6500 * 256, 8192 * 256])
def test_large(n):
    A = _banded(n, [-4096, -64, -1, 0, 1, 64, 4096], 4, "const")
    _same(_run(A, 3, 0), _run(A, 3, 0, fused=0))


@pytest.mark.parametrize("diags", [[0], [-1, 0, 1], [-3, 0, 2, 9], [-70, -9, -1, 0, 1, 9, 70], [-5, 1, 0, 7, 8, 9, 11],
                                   [-40, -20, -3, -2, -1, 0, 1, 2], list(range(-3, 4)) + [100, 300]])
@pytest.mark.parametrize("values", ["const", "full"])
@pytest.mark.parametrize("n", [3000, 40000 + 77])
def test_diagonals(diags, values, n):
    """5, 7, up to 8 and up to 16 diagonals, with and without a middle one"""
    A = _banded(n, sorted(diags), 5, values)
    _same(_run(A, 4, 3), _run(A, 4, 3, fused=0))


@pytest.mark.parametrize("grid", [(30, 30, 1), (80, 75, 1), (40, 41, 37)])
@pytest.mark.parametrize("kw", [dict(growth_limit=30.0), dict(growth_limit=0.0), dict(window=16), dict(window=23),
                                dict(max_iter=20), dict(max_iter=41), dict(trace=True), dict(x_zero=True),
                                dict(growth_limit=30.0, window=40)])
def test_windows_and_switches(grid, kw):
    """every seed but the slowest switches; a low growth limit closes windows
    in the middle of a launch's iterations"""
    nx, ny, nz = grid
    A = P.conv_diff_3d(nx, ny, nz) if nz > 1 else P.conv_diff_2d(nx, ny, 4.01)
    for seed in (0, 6):
        _same(_run(A, 9, seed, **kw), _run(A, 9, seed, fused=0, **kw))


def test_many_shifts():
    """more shifts than the stage has threads"""
    A = P.conv_diff_2d(40, 40, 4.01)
    _same(_run(A, 1100, 900), _run(A, 1100, 900, fused=0))


@pytest.mark.parametrize("x_zero", [True, False])
@pytest.mark.parametrize("n", [7, 16, 33, 1000, 4096 + 65, 43700 + 1, 65536 + 17, 131072 + 63])
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 65])
def test_flush_chunks(M, n, x_zero):
    """The flush on the matrix cores (16 shifts a chunk, 16 to 64 elements a
    wave) against the vector flush of the launches: a last chunk of one or 16
    shifts, and the sizes around which the shapes of its waves change."""
    A = _banded(n, [-2, 0, 1], 5, "const")
    kw = dict(window=6, growth_limit=30.0, x_zero=x_zero)
    _same(_run(A, M, 0, fused=1, **kw), _run(A, M, 0, fused=0, **kw))


@pytest.mark.parametrize("M", [7, 300])
@pytest.mark.parametrize("seed", [0, 5])
def test_hand_over(M, seed):
    """a resident launch that finds its workgroups missing leaves the solve to
    the launch-per-phase kernels (M: with the scalar stage in the shift
    kernel and in a launch of its own)"""
    A = P.conv_diff_2d(90, 81, 4.01)
    _same(_run(A, M, seed, fused=4), _run(A, M, seed, fused=0))


def _batch(mats, **kw):
    """Two solves of a batch of matrices, problem i with 1 + 5 i mod 37 shifts."""
    dev = "cuda"
    spec = []
    for i, A in enumerate(mats):
        M = 1 + 5 * i % 37
        spec.append({"val": torch.as_tensor(A.val).to(dev), "col": torch.as_tensor(A.col.view(np.int32)).to(dev),
                     "ptr": torch.as_tensor(A.ptr.view(np.int32)).to(dev),
                     "b": torch.as_tensor(P.uniform(i, 1, A.n, -1.0, 1.0)).to(dev),
                     "sigma": P.logspace_shifts(M, 1e-3, 1.0), "seed": M // 2 if i % 3 else 0})
    bt = Batch(None, make_params(tol=1e-10, graph=1, **kw), device_spec=spec)
    out = []
    for _ in range(2):
        k, xs, _ = bt.solve()
        for i in range(len(mats)):
            rep, stop, sw = bt.report(i)
            out.append((int(k[i]), xs[i].clone(), torch.zeros(1), stop.copy(), list(sw), rep["status"], None))
    bt.close()
    return out


_T = 256


@pytest.mark.parametrize("kw", [{}, dict(window=17, growth_limit=30.0), dict(fused=4), dict(window=9)])
@pytest.mark.parametrize("sizes", [
    [1, 63, 256, 257, 1000, 4 * _T, 4 * _T + 3, 16 * _T, 16 * _T + 1],        # one workgroup, and the first of two
    [17 * _T - 1, 63 * _T + 77, 64 * _T, 255 * _T, 256 * _T + 9, 20 * _T],    # one tile a column, and one more
    [513 * _T - 100, 300 * _T, 900 * _T + 1, 1024 * _T, 600 * _T],            # up to four
    [1025 * _T, 2048 * _T - 1, 100 * _T, 2],                                  # up to eight
    [2049 * _T, 100 * _T, 2],                                                 # one that does not fit
])
def test_batch(sizes, kw):
    """clusters of one to many workgroups (all sizes of their columns), next
    to each other; more of them than compute units"""
    mats = [_banded(n, ([0], [-1, 0, 1], [-7, -1, 0, 1, 7], [-40, -6, -1, 0, 1, 6, 40],
                        [-5, 1, 0, 7, 8, 9, 11, 300])[i % 5] if n > 300 else [-1, 0, 1], i,
                    "full" if i % 2 else "const") for i, n in enumerate(sizes)]
    _same(_batch(mats, **kw), _batch(mats, **{**kw, "fused": 0}))


def test_batch_more_clusters_than_compute_units():
    mats = [P.conv_diff_2d(60 + i % 50, 70, 4.01) for i in range(320)]
    _same(_batch(mats), _batch(mats, fused=0))


def test_values_in_place():
    """value_index = 0: the values are read at every solve"""
    A = P.conv_diff_3d(20, 21, 22)
    dev = "cuda"
    t = [torch.as_tensor(A.val).to(dev), torch.as_tensor(A.col.view(np.int32)).to(dev),
         torch.as_tensor(A.ptr.view(np.int32)).to(dev)]
    b = torch.as_tensor(P.uniform(1, 1, A.n, -1.0, 1.0)).to(dev)
    pl = Plan(None, 3, make_params(tol=1e-10, graph=1, value_index=False), tensors=t)
    sig = P.logspace_shifts(3, 1e-2, 1.0)
    pl.solve(b, sig, 0)
    t[0].mul_(1.5)
    _, x, _ = pl.solve(b, sig, 0)
    fresh = Plan(None, 3, make_params(tol=1e-10, graph=1, value_index=False, fused=0), tensors=t)
    _, want, _ = fresh.solve(b, sig, 0)
    assert torch.equal(x, want)


def test_memory_kept_between_plans():
    """plans that follow each other run on the memory of those before, from
    two threads too, and give the same results"""
    import threading

    from hbicg import _lib
    A, B = P.conv_diff_2d(70, 60, 4.01), P.conv_diff_3d(25, 24, 23)
    want = {id(A): _run(A, 6, 0, fused=0), id(B): _run(B, 6, 0, fused=0)}
    got = []

    def turns(order):
        for M in order:
            got.append((id(M), _run(M, 6, 0)))

    ts = [threading.Thread(target=turns, args=(o,)) for o in ((A, B, A, B), (B, B, A, A))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    _lib.load().hbicg_trim()
    turns((A, B))
    assert len(got) == 10
    for key, g in got:
        _same(g, want[key])
