"""SGS / ILU(0) sweeps by pencils (5- and 7-point grids) against the oracle's
sequential loops, bit for bit: cross-sections cut at the far faces, lines
shorter than the skew, one pencil and many, both precisions, rows the fast
division does not cover, special values, and patterns that must not take the
pencils."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 1), (63, 66, 1), (40, 300, 1), (200, 129, 1),    # 2D: one pencil, a cut one, short lines
          (16, 16, 16), (17, 19, 23), (8, 32, 40), (100, 9, 7), (33, 64, 8)]


def system(pkg, shape, upwind=True):
    nx, ny, nz = shape
    if upwind:
        return pkg.problem(pkg.UPWIND_CONVDIFF, nx, ny, nz, p0=1e-2, p1=5.0, seed=4)
    return pkg.problem(pkg.FV_DIFFUSION, nx, ny, nz, p0=1.0, seed=4)


def same(a, b):
    return np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a[a == 0]), np.signbit(b[b == 0]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_pencils_bitwise(pkg, oracle, ctx, shape, dtype):
    row, col, val, rhs = system(pkg, shape)
    n = len(rhs)
    rhs = rhs.astype(dtype)
    rhs[::5] = 0
    rhs[3] = -0.0
    lu = pkg.ilu0_factor(row, col, val).astype(dtype)
    for kind, v, ref in (("sgs", val.astype(dtype), oracle.sgs), ("ilu0", lu, oracle.ilu_solve)):
        A = pkg.CsrMatrix(ctx, row, col, v)
        M = getattr(pkg.Preconditioner, kind)(A, row, col)
        print(f"pencils {shape} {kind} {np.dtype(dtype).name}: {M.sweep_blocks()}", flush=True)
        assert M.sweep_blocks()[0] == -(-shape[1] // (64 if shape[2] == 1 else 8)) * -(-shape[2] // 8)
        X, Y = pkg.Vector(ctx, rhs, dtype), pkg.Vector(ctx, n, dtype)
        for waves in (0, 0, 1):
            M.set_sweep(pkg.SWEEP_SYNCFREE, waves)
            M.apply(X, Y)
            M.sweep_status()
            assert same(Y.numpy(), ref(oracle.Csr(row, col, v), rhs))
        # new values reach the sweeps' copies
        v2 = (v * np.random.default_rng(1).uniform(0.5, 1.5, len(v))).astype(dtype)
        A.upload_values(v2)
        M.apply(X, Y)
        assert same(Y.numpy(), ref(oracle.Csr(row, col, v2), rhs))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(70, 66, 1), (18, 17, 16)])
def test_pencils_division_and_special_values(pkg, oracle, ctx, shape, dtype):
    """Diagonals and results outside the range of the fast division, values
    that overflow, infinities and NaN in the right-hand side."""
    row, col, val, rhs = system(pkg, shape, upwind=False)
    n = len(rhs)
    big = 2.0 ** (350 if dtype == np.float64 else 45)
    tiny = 2.0 ** (-560 if dtype == np.float64 else -70)
    bad = rhs.astype(dtype).copy()
    bad[n // 2], bad[n // 3], bad[n - 1] = np.inf, -np.inf, np.nan
    far = rhs.astype(dtype).copy()
    far[n - 1] = np.inf        # the far end: reaches every row of the backward sweep that depends on it
    cases = [(val, rhs * tiny), (val * big, rhs), (val / big, rhs), (val, bad), (val, far)]
    for v, b in cases:
        v, b = v.astype(dtype), np.asarray(b).astype(dtype)
        A = pkg.CsrMatrix(ctx, row, col, v)
        M = pkg.Preconditioner.sgs(A, row, col)
        assert M.sweep_blocks()[0] > 0
        Y = pkg.Vector(ctx, n, dtype)
        M.apply(pkg.Vector(ctx, b, dtype), Y)
        M.sweep_status()
        with np.errstate(all="ignore"):
            assert same(Y.numpy(), oracle.sgs(oracle.Csr(row, col, v), b))


@pytest.mark.parametrize("what", ["missing", "periodic", "rows"])
def test_other_patterns_keep_their_schedule(pkg, oracle, ctx, what):
    """A grid with an entry missing, one with a wrapped neighbour and one whose
    row count is no multiple of the line take the other schedules."""
    nx, ny = 70, 66
    row, col, val, rhs = system(pkg, (nx, ny, 1))
    n = len(rhs)
    D = {(i, int(c)): v for i in range(n) for c, v in zip(col[row[i]:row[i + 1]], val[row[i]:row[i + 1]])}
    if what == "missing":
        del D[(nx * 9 + 7, nx * 9 + 6)]
    elif what == "periodic":
        D[(nx * 9, nx * 9 - 1)] = -0.25
    else:
        n -= 5
        D = {k: v for k, v in D.items() if k[0] < n and k[1] < n}
    keys = sorted(D)
    row = np.searchsorted([k[0] for k in keys], np.arange(n + 1)).astype(np.int32)
    col = np.array([k[1] for k in keys], np.int32)
    val = np.array([D[k] for k in keys])
    rhs = rhs[:n]
    A = pkg.CsrMatrix(ctx, row, col, val)
    M = pkg.Preconditioner.sgs(A, row, col)
    assert M.sweep_blocks()[0] != -(-ny // 64)   # two pencils otherwise
    Y = pkg.Vector(ctx, n)
    M.apply(pkg.Vector(ctx, rhs), Y)
    assert np.array_equal(Y.numpy(), oracle.sgs(oracle.Csr(row, col, val), rhs))


@pytest.mark.parametrize("shape", [(70, 66, 1), (18, 17, 16)])
@pytest.mark.parametrize("limit", [1, 4096])
def test_no_room_for_the_pencils(pkg, oracle, ctx, shape, limit):
    """Without memory for the first or a later one of the pencils' copies the
    preconditioner is created all the same and sweeps by blocks."""
    row, col, val, rhs = system(pkg, shape)
    A = pkg.CsrMatrix(ctx, row, col, val)
    ctx.set_copy_limit(limit)
    try:
        M = pkg.Preconditioner.sgs(A, row, col)
    finally:
        ctx.set_copy_limit(0)
    pencils = pkg.Preconditioner.sgs(A, row, col).sweep_blocks()
    assert M.sweep_blocks()[0] > pencils[0] > 0
    Y = pkg.Vector(ctx, len(rhs))
    M.apply(pkg.Vector(ctx, rhs), Y)
    M.sweep_status()
    assert same(Y.numpy(), oracle.sgs(oracle.Csr(row, col, val), rhs))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape, bound", [((8, 260, 260), 1089), ((70, 300 * 64 - 7, 1), 300)])
def test_more_pencils_than_workgroups(pkg, oracle, ctx, shape, bound, dtype):
    """One workgroup per compute unit and several pencils for each: the tickets,
    the LDS ring cleared between pencils, the counters handed from sweep to
    sweep and the inboxes emptied for the next apply."""
    row, col, val, rhs = system(pkg, shape)
    val, rhs = val.astype(dtype), rhs.astype(dtype)
    A = pkg.CsrMatrix(ctx, row, col, val)
    M = pkg.Preconditioner.sgs(A, row, col)
    assert M.sweep_blocks()[0] == bound > ctx.info()["num_cu"]
    M.set_sweep(pkg.SWEEP_SYNCFREE, 1)
    want = oracle.sgs(oracle.Csr(row, col, val), rhs)
    X, Y = pkg.Vector(ctx, rhs, dtype), pkg.Vector(ctx, len(rhs), dtype)
    for _ in range(4):
        Y.zeros()
        M.apply(X, Y)
        M.sweep_status()
        assert same(Y.numpy(), want)
    # another right-hand side meets nothing of the last one
    X.scale(-2.0)
    M.apply(X, Y)
    assert same(Y.numpy(), -2 * want)
