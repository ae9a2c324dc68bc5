"""SpMV from (offset, value) pairs against the slot-pair layout of the same
matrix, bit for bit: grids cut at every side, one and several slices, rows
whose window leaves x, a full and a one-too-long list of pairs, values that
change, and matrices that must keep the general layouts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def stencil(shape, offsets, values, diag=None):
    """Constant-coefficient stencil on a grid, entries outside left out."""
    idx = np.indices(shape).reshape(len(shape), -1).T
    n = len(idx)
    stride = np.cumprod([1] + list(shape[::-1]))[:-1][::-1]
    cols, vals, have = [], [], []
    for o, v in zip(offsets, values):
        t = idx + np.array(o)
        have.append(((t >= 0) & (t < np.array(shape))).all(1))
        cols.append(t @ stride)
        vals.append(np.full(n, v) if any(o) or diag is None else diag)
    cols, vals, have = np.stack(cols, 1), np.stack(vals, 1), np.stack(have, 1)
    order = np.argsort(cols, 1)
    cols, vals, have = (np.take_along_axis(a, order, 1) for a in (cols, vals, have))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(have.sum(1), out=row[1:])
    return row, cols[have].astype(np.int32), vals[have]


def box(dim):
    o = np.indices((3,) * dim).reshape(dim, -1).T - 1
    return o, 0.1 + np.abs(o).sum(1) / 3.0


def cross(dim):
    o = np.concatenate([np.zeros((1, dim), int), np.eye(dim, dtype=int), -np.eye(dim, dtype=int)])
    return o, np.array([2.0 * dim + 0.3] + [-1.0 / 3] * dim + [-0.7] * dim)


def compare(pkg, ctx, row, col, val, dtype, pairs, ncol=None, x=None):
    n = len(row) - 1
    ncol = n if ncol is None else ncol
    val = val.astype(dtype)
    A = pkg.CsrMatrix(ctx, row, col, val, ncol=ncol)
    B = pkg.CsrMatrix(ctx, row, col, val, ncol=ncol)
    B.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
    assert (pairs is None or A.pattern_pairs() == pairs) and B.pattern_pairs() == 0
    rng = np.random.default_rng(n)
    x = rng.standard_normal(ncol) if x is None else x
    y0 = rng.standard_normal(n)
    X = pkg.Vector(ctx, x, dtype)
    for add in (False, True):
        Y, Z = pkg.Vector(ctx, y0, dtype), pkg.Vector(ctx, y0, dtype)
        (A.spmv_add if add else A.spmv)(X, Y)
        (B.spmv_add if add else B.spmv)(X, Z)
        assert np.array_equal(Y.numpy(), Z.numpy(), equal_nan=True)
    return A


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(1, 1, 64), (4, 4, 4), (6, 8, 16), (5, 9, 31), (7, 20, 63), (11, 6, 64), (9, 33, 65)])
def test_grids(pkg, ctx, shape, dtype):
    big = shape != (4, 4, 4)     # a slice of mostly boundary rows: padding rules the layout out
    compare(pkg, ctx, *stencil(shape, *box(3)), dtype, (27 if min(shape) > 1 else 3) if big else None)
    compare(pkg, ctx, *stencil(shape[1:], *box(2)), dtype, (9 if shape[1] > 1 else 3) if big else None)
    compare(pkg, ctx, *stencil(shape, *cross(3)), dtype, (7 if min(shape) > 1 else 3) if big else None)
    compare(pkg, ctx, *stencil(shape[1:], *cross(2)), dtype, (5 if shape[1] > 1 else 3) if big else None)


@pytest.mark.parametrize("k", [1, 2, 3])
def test_values_per_row(pkg, ctx, k):
    """k values of the diagonal; a third one lies between the sampled rows."""
    n = 20 * 21 * 22
    d = 5.0 + (np.arange(n) * k // n)
    compare(pkg, ctx, *stencil((20, 21, 22), *cross(3), diag=d), np.float64, 6 + k if k <= 2 else None)
    i = np.arange(k * 128)
    compare(pkg, ctx, np.arange(len(i) + 1, dtype=np.int32), i.astype(np.int32), 1.0 + i // 128, np.float64,
            k if k <= 2 else 0)


@pytest.mark.parametrize("width", [31, 32, 33])
def test_longest_list(pkg, ctx, width):
    """A set holds 32 pairs; longer rows take the general layout."""
    n = 700
    c = np.arange(n)[:, None] + np.arange(width) - 5
    m = (c >= 0) & (c < n)
    v = np.broadcast_to(np.cos(np.arange(width)), c.shape)
    row = np.zeros(n + 1, np.int32)
    np.cumsum(m.sum(1), out=row[1:])
    for dtype in (np.float64, np.float32):
        compare(pkg, ctx, row, c[m].astype(np.int32), v[m], dtype, width if width <= 32 else 0)


@pytest.mark.parametrize("reach", [1, 63, 64, 500, 1999])
def test_windows_and_rectangles(pkg, ctx, reach):
    n = 2000
    for ncol in (n, n + 300, n - 300):
        r = np.repeat(np.arange(n), 3)
        c = (np.arange(n)[:, None] + np.array([-reach, 0, reach])).ravel()
        v = np.tile([0.5, -0.25, 3.0], n)
        m = (c >= 0) & (c < ncol)
        row = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(r[m], minlength=n), out=row[1:])
        compare(pkg, ctx, row, c[m].astype(np.int32), v[m], np.float64, len(set(zip(c[m] - r[m], v[m]))), ncol=ncol)


def test_entries_left_out_are_not_read_into_sums(pkg, ctx):
    """Infinities and NaN of x reach only the rows that hold their columns."""
    row, col, val = stencil((9, 33, 65), *box(3))
    x = np.random.default_rng(0).standard_normal(len(row) - 1)
    x[::97] = np.inf
    x[5::101] = np.nan
    x[7::89] = -0.0
    compare(pkg, ctx, row, col, val, np.float64, 27, x=x)


def test_values_change(pkg, ctx):
    row, col, val = stencil((12, 13, 70), *box(3))
    A = compare(pkg, ctx, row, col, val, np.float64, 27)
    x = np.random.default_rng(1).standard_normal(len(row) - 1)
    X, Y = pkg.Vector(ctx, x), pkg.Vector(ctx, len(x))
    for v in (val * np.random.default_rng(2).uniform(1, 2, len(val)), np.where(np.arange(len(val)) == 4321, 9.0, val), val * 2):
        B = pkg.CsrMatrix(ctx, row, col, v)
        B.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
        Z = pkg.Vector(ctx, len(x))
        A.upload_values(v)
        A.spmv(X, Y)
        B.spmv(X, Z)
        assert np.array_equal(Y.numpy(), Z.numpy())
    assert A.pattern_pairs() == 27
    assert pkg.CsrMatrix.cast_of(A, np.float32).pattern_pairs() == 27
    A.swap_diag_front()      # the row order is no longer ascending
    assert A.pattern_pairs() == 0


def test_no_room_for_the_list(pkg, ctx):
    """Without memory for the list every call that would make it succeeds in
    the general layout: upload, new values, another layout and back, a cast."""
    shape = (12, 13, 70)
    row, col, val = stencil(shape, *box(3))
    ctx.set_copy_limit(1)
    try:
        A = compare(pkg, ctx, row, col, val, np.float64, 0)
        A.upload_values(2 * val)
        A.scale(0.5)
        A.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
        A.set_spmv(pkg.SPMV_AUTO)
        assert A.pattern_pairs() == 0 and pkg.CsrMatrix.cast_of(A, np.float32).pattern_pairs() == 0
    finally:
        ctx.set_copy_limit(0)
    A.upload_values(val)
    assert A.pattern_pairs() == 27


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_pairs_that_few_rows_hold(pkg, ctx, dtype):
    """Pairs of single rows far from the probed ones are found in later rounds,
    at the first and the last row of a slice and in the last, cut slice; a list
    that grows past a set, and one most rows hold little of, is not taken."""
    shape = (9, 33, 65)
    row, col, val = stencil(shape, *box(3))
    n = len(row) - 1
    for rows, pairs in (([64 * 50], 28), ([63], 28), ([n - 1], 28), ([64 * 7, 64 * 9 + 63, n - 2], 30),
                        (list(range(70, 70 + 64 * 5, 64)), 32), (list(range(70, 70 + 64 * 6, 64)), 0)):
        v = val.copy()
        for i, r in enumerate(rows):
            v[row[r] + np.flatnonzero(col[row[r]:row[r + 1]] == r)] = 20.0 + i
        compare(pkg, ctx, row, col, v, dtype, pairs)
    # 3 of 12 / 16 pairs per row
    for k in (12, 16):
        i, rng = np.arange(4000), np.random.default_rng(k)
        o = np.sort(np.argsort(rng.random((4000, k)), 1)[:, :3], 1) * 7
        c = i[:, None] + o
        m = c < 4000
        r = np.zeros(4001, np.int32)
        np.cumsum(m.sum(1), out=r[1:])
        compare(pkg, ctx, r, c[m].astype(np.int32), np.cos(o[m]), dtype, k if 4 * m.sum() >= k * 4000 else 0)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("what", ["box", "cross", "two diagonals", "band"])
def test_scaled_values(pkg, ctx, what, dtype):
    """Scaling keeps the pairs and their rounding: the whole matrix, the entries
    off the diagonal, a factor that rounds, one that makes pairs equal (0), and
    new values afterwards."""
    shape = (12, 13, 70)
    if what == "band":      # offsets whose runs start, centre and end at 0
        n = 700
        c = np.arange(n)[:, None] + np.array([-9, -2, -1, 0, 1, 2, 40])
        m = (c >= 0) & (c < n)
        row, col, val = np.concatenate([[0], np.cumsum(m.sum(1))]).astype(np.int32), c[m].astype(np.int32), \
            np.broadcast_to(np.cos(np.arange(7)), c.shape)[m]
    elif what == "two diagonals":
        n = 12 * 13 * 70
        row, col, val = stencil(shape, *cross(3), diag=5.0 + (np.arange(n) * 2 // n))
    else:
        row, col, val = stencil(shape, *(box(3) if what == "box" else cross(3)))
    n = len(row) - 1
    A, B = pkg.CsrMatrix(ctx, row, col, val, dtype=dtype), pkg.CsrMatrix(ctx, row, col, val, dtype=dtype)
    B.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
    pairs = A.pattern_pairs()
    assert pairs > 0 and B.pattern_pairs() == 0
    X, Y, Z = pkg.Vector(ctx, np.random.default_rng(3).standard_normal(n), dtype), pkg.Vector(ctx, n, dtype), pkg.Vector(ctx, n, dtype)
    for alpha, off in ((-1.0 / 3, False), (0.1, True), (1e-30, False), (1e30, True), (0.0, True), (7.0, False), (0.0, False)):
        A.scale(alpha, off)
        B.scale(alpha, off)
        assert A.pattern_pairs() == pairs
        A.spmv(X, Y)
        B.spmv(X, Z)
        assert np.array_equal(Y.numpy(), Z.numpy())
    A.upload_values(val.astype(dtype))
    B.upload_values(val.astype(dtype))
    A.spmv(X, Y)
    B.spmv(X, Z)
    assert A.pattern_pairs() == pairs and np.array_equal(Y.numpy(), Z.numpy()) and Y.nrm2() > 0
