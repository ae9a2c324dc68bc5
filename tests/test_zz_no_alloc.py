"""The allocation-free CG (hfh_pcg_solve_noalloc) against hfh_pcg_solve.

Both run the same kernels in the same order; the allocation-free one keeps
its work space in the library's static device array, starts the one-launch
form with a plain launch instead of a cooperative one and the launched form's
loop directly instead of through a graph.  So iterates, histories, states and
solutions are bit-identical in both forms.  Two calls in a row, the second on a smaller
system, check that nothing of the first call's contents survives into the
second; the size limit and the preconditioner restriction are checked as
errors."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _both(pkg, ctx, row, col, val, rhs, dtype, prec, form, maxits=3000, rtol=1e-8):
    """form: "one launch" (the automatic layout of a system that fits on the
    chip) or "launched" (an explicit layout rules the one launch out)."""
    out = []
    for noalloc in (False, True):
        A = pkg.CsrMatrix(ctx, row, col, val, dtype=dtype)
        if form == "launched":
            A.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
        ran = ctx.cg_launches()[0]
        P = pkg.Preconditioner.jacobi(A) if prec else None
        X = pkg.Vector(ctx, len(rhs), dtype)
        info = pkg.pcg(A, pkg.Vector(ctx, rhs, dtype), X, P, maxits=maxits, atol=0.0, rtol=rtol, history=True,
                       noalloc=noalloc)
        assert ctx.cg_launches()[0] - ran == (form == "one launch")
        out.append((info, X.numpy()))
    return out


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("prec", [True, False])
@pytest.mark.parametrize("form", ["one launch", "launched"])
def test_noalloc_equals_allocating_entry(pkg, ctx, dtype, prec, form):
    # first a 3D Q1 system (the larger with two rows of 27 entries per thread),
    # then a smaller 2D one on the same static array
    for kind, m in ((pkg.Q1_3D, 31), (pkg.Q1_3D, 54), (pkg.Q1_2D, 40)):
        row, col, val, rhs = pkg.problem(kind, m)
        (ia, xa), (ib, xb) = _both(pkg, ctx, row, col, val, rhs, dtype, prec, form)
        print(f"noalloc case dtype={np.dtype(dtype).name} jacobi={prec} n={len(rhs)}: iters {ia['iters']} / "
              f"{ib['iters']}", flush=True)
        assert ia["state"] == pkg.SUCCESS_REL
        assert ib["state"] == ia["state"]
        assert ib["iters"] == ia["iters"]
        assert ib["res"] == ia["res"] and ib["res0"] == ia["res0"]
        assert np.array_equal(ib["hist"], ia["hist"])
        assert np.array_equal(xb, xa)


@pytest.mark.parametrize("form", ["one launch", "launched"])
def test_noalloc_maxits_state(pkg, ctx, form):
    """A solve stopped by maxits reports the same state and iterate."""
    row, col, val, rhs = pkg.problem(pkg.FV_DIFFUSION, 12, p0=1.0, seed=2)
    res = []
    for noalloc in (False, True):
        A = pkg.CsrMatrix(ctx, row, col, val)
        if form == "launched":
            A.set_spmv(pkg.SPMV_SELL_PAIRS, 1)
        X = pkg.Vector(ctx, len(rhs))
        info = pkg.pcg(A, pkg.Vector(ctx, rhs), X, pkg.Preconditioner.jacobi(A), maxits=7, atol=0.0, rtol=1e-12,
                       check=False, noalloc=noalloc)
        res.append((info, X.numpy()))
    (ia, xa), (ib, xb) = res
    assert ia["state"] == pkg.FAIL_MAXITS == ib["state"]
    assert ia["iters"] == ib["iters"] == 7
    assert np.array_equal(xa, xb)


def test_noalloc_limits(pkg, ctx):
    """Beyond the static array: HFH_ERR_INVALID before any launch; an
    MC-SGS preconditioner: HFH_ERR_UNSUPPORTED.  The same diagonal system in
    FP32 fits and is solved in one step."""
    n = 2_200_000   # FP64: 4 vectors of 17.6 MB exceed the 64 MiB array
    row = np.arange(n + 1, dtype=np.int32)
    col = np.arange(n, dtype=np.int32)
    val = np.full(n, 2.0)
    rhs = np.ones(n)
    A = pkg.CsrMatrix(ctx, row, col, val)
    X = pkg.Vector(ctx, n)
    ctl = pkg.Control(10, 0.0, 1e-8, 1e6)
    inf = pkg.SolveInfo()
    B = pkg.Vector(ctx, rhs)   # kept alive through the call
    rc = pkg.hip().hfh_pcg_solve_noalloc(A.h, None, B.h, X.h, C.byref(ctl), C.byref(inf), None)
    assert rc == pkg.ERR_INVALID
    assert "static" in pkg.hip().hfh_last_error().decode()
    Af = pkg.CsrMatrix(ctx, row, col, val, dtype=np.float32)
    Xf = pkg.Vector(ctx, n, np.float32)
    info = pkg.pcg(Af, pkg.Vector(ctx, rhs, np.float32), Xf, None, maxits=10, atol=0.0, rtol=1e-6, noalloc=True)
    assert info["iters"] == 1
    assert np.array_equal(Xf.numpy(), np.full(n, 0.5, np.float32))
    # MC-SGS is refused
    row2, col2, val2, rhs2 = pkg.problem(pkg.FV_DIFFUSION, 8, p0=1.0, seed=1)
    nc, color, sizes, perm = pkg.multicoloring(row2, col2)
    prow, pcol, pval = pkg.csr_permute(row2, col2, val2, perm)
    A2 = pkg.CsrMatrix(ctx, prow, pcol, pval)
    P2 = pkg.Preconditioner.mcsgs(A2, sizes)
    with pytest.raises(pkg.HfhError):
        pkg.pcg(A2, pkg.Vector(ctx, rhs2[perm]), pkg.Vector(ctx, len(rhs2)), P2, noalloc=True)


CHILD = r"""
import ctypes as C, sys
sys.path.insert(0, "tests")
from conftest import load_pkg
P = load_pkg()
kind, m, form = sys.argv[1], int(sys.argv[2]), sys.argv[3]
ctx = P.Context(0)
row, col, val, rhs = P.problem(getattr(P, kind), m)
A = P.CsrMatrix(ctx, row, col, val)
if form == "launched":
    A.set_spmv(P.SPMV_SELL_PAIRS, 1)
M, B, X = P.Preconditioner.jacobi(A), P.Vector(ctx, rhs), P.Vector(ctx, len(rhs))
hip = C.CDLL("libamdhip64.so")


def free():
    ctx.sync()
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


A.spmv(B, X)
B.dot(X)          # the vector kernels' code is loaded by the first of them
X.zeros()
before = free()
P.pcg(A, B, X, M, maxits=50, atol=0.0, rtol=1e-8, check=False, noalloc=True)
after = free()
assert ctx.cg_launches() == ((0, 0) if form == "launched" else (1, 0)), ctx.cg_launches()
print("USED", before - after)
"""


@pytest.mark.parametrize("kind, m, form", [("Q1_3D", 10, "one launch"), ("Q1_3D", 56, "one launch"),
                                           ("Q1_2D", 256, "one launch"), ("Q1_2D", 256, "launched")])
def test_first_solve_of_a_process_allocates_nothing(kind, m, form):
    """Neither the library nor the runtime (scratch of a kernel with spilled
    registers, the queue of cooperative launches) takes device memory."""
    r = subprocess.run([sys.executable, "-c", CHILD, kind, str(m), form], cwd=ROOT, capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    print(f"noalloc memory {kind} {m} {form}: {r.stdout.strip()}", flush=True)
    assert r.stdout.split("USED")[1].strip() == "0"
