"""CG in one launch (systems that fit on the chip) against the oracle's CG, at
the sizes where its layout changes: one workgroup and several, one, two and
four rows per thread, every bound of the row length, windows cut at both ends
of the matrix, and the systems that must take the launched form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banded(n, half, reach, seed=0):
    """SPD: up to 2 half + 1 entries per row at distances up to `reach`."""
    rng = np.random.default_rng(seed)
    dist = np.unique(np.concatenate([[1], np.linspace(1, reach, half).astype(int)]))[:half] if half else np.array([], int)
    rows, cols, vals = [np.arange(n)], [np.arange(n)], []
    diag = np.full(n, 0.1)
    for d in dist:
        if d >= n:
            continue
        w = rng.uniform(0.1, 1.0, n - d)
        i = np.arange(n - d)
        rows += [i, i + d]
        cols += [i + d, i]
        vals += [-w, -w]
        diag[:n - d] += w
        diag[d:] += w
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate([diag] + vals)
    o = np.lexsort((c, r))
    row = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=row[1:])
    return row, c[o].astype(np.int32), v[o], rng.standard_normal(n)


def check(pkg, oracle, ctx, system, dtype=np.float64, prec=True, x0=None, one=True, **kw):
    """one: the solve must be one launch (True) or must not be (False)."""
    row, col, val, rhs = system
    val, rhs = val.astype(dtype), rhs.astype(dtype)
    n = len(rhs)
    ctl = dict(maxits=2000, atol=0.0, rtol=1e-8 if dtype == np.float64 else 1e-4, dtol=1e6)
    ctl.update(kw)
    A = pkg.CsrMatrix(ctx, row, col, val)
    M = pkg.Preconditioner.jacobi(A) if prec else None
    X = pkg.Vector(ctx, np.zeros(n) if x0 is None else x0, dtype)
    ran = ctx.cg_launches()
    info = pkg.pcg(A, pkg.Vector(ctx, rhs, dtype), X, M, history=True, check=False, **ctl)
    assert ctx.cg_launches() == (ran[0] + one, ran[1])
    OA = oracle.Csr(row, col, val)
    xo, oi = oracle.cg(OA, rhs, x0=None if x0 is None else x0.astype(dtype), P=oracle.Prec.jacobi(OA) if prec else None,
                       ctrl=(ctl["maxits"], ctl["atol"], ctl["rtol"], ctl["dtol"]))
    assert info["state"] == oi["status"]
    assert abs(info["iters"] - oi["iters"]) <= 2
    k = min(12, len(info["hist"]), len(oi["hist"]))
    # each step rounds a residual vector of up to the largest norm so far, so
    # after k <= 12 steps the norms differ by up to about 12 eps of it
    floor = 12 * np.finfo(dtype).eps * np.max(oi["hist"][:k])
    assert np.allclose(info["hist"][:k], oi["hist"][:k], rtol=1e-9 if dtype == np.float64 else 1e-4, atol=floor)
    if info["state"] in (pkg.SUCCESS_ABS, pkg.SUCCESS_REL):
        # the recursive residual met the test; the true one differs by the
        # rounding of x and r, far below twice the tolerances used here
        goal = max(ctl["atol"], ctl["rtol"] * info["res0"])
        r = rhs.astype(np.float64) - oracle.spmv(oracle.Csr(row, col, val.astype(np.float64)), X.numpy().astype(np.float64))
        assert np.linalg.norm(r) <= (2 if dtype == np.float64 else 10) * goal
    return info, X.numpy()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 63, 511, 512, 513, 1024, 1025, 2048, 2049, 2560, 2561, 131072, 131073, 262145,
                               524288, 524289])
def test_sizes(pkg, oracle, ctx, n, dtype):
    check(pkg, oracle, ctx, banded(n, 2, min(40, max(1, n - 1)), seed=n), dtype, one=n <= 4 * 512 * ctx.info()["num_cu"])


@pytest.mark.parametrize("half", [0, 1, 2, 3, 4, 5, 7, 8, 13, 14])
@pytest.mark.parametrize("n", [700, 1500, 6000])
def test_row_lengths(pkg, oracle, ctx, n, half):
    """2 half + 1 entries: 5, 7, 9, 16 and 28 bound the kernels; 29 takes the launches."""
    for prec in (True, False):
        check(pkg, oracle, ctx, banded(n, half, 300, seed=half), prec=prec, one=half <= 13)


def launches(n, half, reach, size):
    """Does CG on banded(n, half, reach) take one launch?  Its workgroups' rows,
    the reach on both sides and a zero must fit 158 KiB of LDS, and the far rows
    must not take longer than the launches."""
    rows = 512 * next(e for e in (1, 2, 4) if n <= 512 * 256 * e)
    far = min(rows + 2 * reach, n) - rows
    length = 2 * half + 1
    limit = 65536 if length > 16 else 21000 if rows < 2048 else 28000 if length <= 5 else 34000
    return (rows + far + 1) * size <= 158 * 1024 and far <= limit


@pytest.mark.parametrize("n, half, reach, one64, one32", [
    (40000, 2, 9000, True, True),       # near the LDS size in FP64
    (20000, 2, 19999, True, True),      # as long as the matrix
    (40000, 2, 10500, False, True), (40000, 2, 10501, False, False),    # the far rows
    (40000, 2, 39999, False, False), (140000, 4, 10501, False, False),
    (270000, 2, 14000, False, True), (270000, 2, 14001, False, False),
    (270000, 4, 17000, False, True), (270000, 4, 17001, False, False),
    (40000, 9, 15000, False, True), (40000, 9, 19000, False, True)])
def test_windows(pkg, oracle, ctx, n, half, reach, one64, one32):
    """Windows near the LDS size, beyond it (launched form), as long as the
    matrix, and with more far rows than pay."""
    if ctx.info()["num_cu"] >= 256:
        assert (launches(n, half, reach, 8), launches(n, half, reach, 4)) == (one64, one32)
    check(pkg, oracle, ctx, banded(n, half, reach, seed=1), one=one64)
    check(pkg, oracle, ctx, banded(n, half, reach, seed=1), np.float32, one=one32)


@pytest.mark.parametrize("n", [1500, 5000])
def test_controls(pkg, oracle, ctx, n):
    s = banded(n, 3, 200, seed=5)
    x0 = np.random.default_rng(9).standard_normal(n)
    check(pkg, oracle, ctx, s, x0=x0)
    assert check(pkg, oracle, ctx, s, maxits=7)[0]["state"] == pkg.FAIL_MAXITS
    assert check(pkg, oracle, ctx, s, atol=1e-3)[0]["state"] == pkg.SUCCESS_ABS
    info, x = check(pkg, oracle, ctx, s, atol=1e6)      # met before the first step
    assert info["iters"] == 0 and not x.any()
    assert check(pkg, oracle, ctx, s, rtol=0.0, maxits=40)[0]["iters"] == 40
    # an indefinite operator may diverge: the same state and step as the oracle
    row, col, val, rhs = s
    check(pkg, oracle, ctx, (row, col, -val, rhs), prec=False)


def test_repeated_and_interleaved(pkg, ctx):
    """Two systems solved in turn, each call's result the same bits."""
    out = {}
    for rep in range(3):
        for n in (3000, 70000):
            row, col, val, rhs = banded(n, 2, 60, seed=n)
            A = pkg.CsrMatrix(ctx, row, col, val)
            X = pkg.Vector(ctx, n)
            pkg.pcg(A, pkg.Vector(ctx, rhs), X, pkg.Preconditioner.jacobi(A), maxits=2000, atol=0.0, rtol=1e-8)
            assert np.array_equal(out.setdefault(n, X.numpy()), X.numpy())


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [5000, 70000])
def test_wait_that_gives_up(pkg, ctx, n, dtype, noalloc):
    """A launch whose waits give up leaves no trace: the launched form solves
    from the initial guess, the same bits as where it is taken at once (per
    SpMV timing rules the one launch out), and the next solve is one launch."""
    row, col, val, rhs = banded(n, 2, 60, seed=n)
    A = pkg.CsrMatrix(ctx, row, col, val.astype(dtype))
    M, B = pkg.Preconditioner.jacobi(A), pkg.Vector(ctx, rhs, dtype)
    x0 = np.random.default_rng(2).standard_normal(n)
    kw = dict(maxits=2000, atol=0.0, rtol=1e-6 if dtype == np.float64 else 1e-4, history=True, check=False, noalloc=noalloc)

    def solve():
        X = pkg.Vector(ctx, x0, dtype)
        before = ctx.cg_launches()
        info = pkg.pcg(A, B, X, M, **kw)
        ran, gave_up = (b - a for a, b in zip(before, ctx.cg_launches()))
        return info, X.numpy(), ran, gave_up

    one = solve()
    assert one[2:] == (1, 0)
    ctx.set_timing(True)
    try:
        want = solve()
    finally:
        ctx.set_timing(False)
    assert want[2:] == (0, 0)
    ctx.set_wait_polls(1)
    try:
        for _ in range(3):
            got = solve()
            assert got[2:] == (0, 1)
            assert got[0]["iters"] == want[0]["iters"] and got[0]["state"] == want[0]["state"]
            assert np.array_equal(got[0]["hist"], want[0]["hist"]) and np.array_equal(got[1], want[1])
    finally:
        ctx.set_wait_polls(0)
    again = solve()
    assert again[2:] == (1, 0) and np.array_equal(again[1], one[1])
