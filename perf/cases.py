"""The workloads whose speed this package is judged by, as data: what a
program that uses the package has it do, over the sizes it does it at.

`listed()` names the fixed cases, `draw(rng)` gives one more case of the same
ranges, `prepare` makes what the program holds before the call (operator,
preconditioner, vectors), `run` is the call, `work` its compulsory traffic and
operations, `tolerance` what another correct implementation may differ by, and
`exact` the same result from plain torch / numpy in 64 bits.

The operators are structured-grid systems of the kinds the package's own
generator, tests and benchmark use, built here with torch:

  q1_2d, q1_3d   Q1 finite element Laplacian on an nx x ny (x nz) interior grid
                 (9 / 27 entries per row), h = 1 / (nx + 1)
  fv             cell-centred finite volume diffusion with lognormal cell
                 coefficients (5 / 7 entries per row, harmonic face means)
  upwind         upwind convection-diffusion with a rotating velocity
                 (5 / 7 entries per row, nonsymmetric)
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _pkg():
    if "hiflow3_amd" not in sys.modules:
        d = os.path.join(_ROOT, "hiflow3_2.0_amd")
        spec = importlib.util.spec_from_file_location("hiflow3_amd", os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["hiflow3_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["hiflow3_amd"]


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = _pkg().Context(0)
    return _ctx


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one SpMV of a small 2D finite element operator (the 256 x 256 mesh):
        # the operand sits in the caches, so latency and the launch count
        {"name": "spmv_q1_2d_255", "do": "spmv", "op": "q1_2d", "nx": 255, "ny": 255, "nz": 1, "f32": False},
        # the package's headline SpMV: the 3D Q1 Laplacian on 128^3 cells
        {"name": "spmv_q1_3d_127", "do": "spmv", "op": "q1_3d", "nx": 127, "ny": 127, "nz": 127, "f32": False},
        # damped Jacobi smoothing (a multigrid smoother's three steps) in single
        # precision on a finite volume operator of uneven size
        {"name": "smooth_fv_3d_f32", "do": "smooth", "op": "fv", "nx": 141, "ny": 118, "nz": 103, "f32": True},
        # the vector part of one step of a host-driven CG (dots that return to
        # the host, axpys, a scaleadd) at 65 thousand unknowns
        {"name": "blas1_65k", "do": "blas1", "op": "none", "nx": 65025, "ny": 1, "nz": 1, "f32": False},
        # a whole small solve: 2D diffusion, 1,517 unknowns, Jacobi-CG
        {"name": "cg_fv_2d_41x37", "do": "cg", "op": "fv", "nx": 41, "ny": 37, "nz": 1, "f32": False},
        # the 2D Q1 Laplacian of the 256 x 256 mesh, Jacobi-CG to 1e-8
        {"name": "cg_q1_2d_255", "do": "cg", "op": "q1_2d", "nx": 255, "ny": 255, "nz": 1, "f32": False},
        # the headline solve: 3D Q1 on 128^3 cells, Jacobi-CG to 1e-8
        {"name": "cg_q1_3d_127", "do": "cg", "op": "q1_3d", "nx": 127, "ny": 127, "nz": 127, "f32": False},
        # variable-coefficient diffusion, CG with multicolour SGS to 1e-10
        {"name": "cgmc_fv_3d_144", "do": "cgmc", "op": "fv", "nx": 144, "ny": 144, "nz": 144, "f32": False},
        # the same kind at 192^3 by mixed precision defect correction to 1e-10
        {"name": "dc_fv_3d_192", "do": "dc", "op": "fv", "nx": 192, "ny": 192, "nz": 192, "f32": False},
        # convection-diffusion on 128^3, GMRES(30) with ILU(0) to 1e-8
        {"name": "gmres_upwind_128", "do": "gmres", "op": "upwind", "nx": 128, "ny": 128, "nz": 128, "f32": False},
        # one symmetric Gauss-Seidel apply on a 2D operator of uneven size
        {"name": "sgs_fv_2d_701x509", "do": "sgs", "op": "fv", "nx": 701, "ny": 509, "nz": 1, "f32": False},
        # the serving engine: 32 diffusion solves of mixed sizes handed in
        # together, FP32 / FP64 CG to 1e-10
        {"name": "serve_32", "do": "serve", "op": "fv", "nmin": 1000, "nmax": 300000, "count": 32, "mix": 7,
         "f32": False},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, n, three, lo=7):
    """nx, ny, nz of about n cells, uneven."""
    d = 3 if three else 2
    side = n ** (1.0 / d)
    nx = max(lo, int(round(side * rng.uniform(0.75, 1.33))))
    ny = max(lo, int(round(side * rng.uniform(0.75, 1.33)))) if three else max(lo, int(n / nx))
    nz = max(lo, int(n / (nx * ny))) if three else 1
    return nx, ny, nz


def draw(rng):
    do = rng.choice(["spmv", "spmv", "smooth", "blas1", "cg", "cg", "cgmc", "dc", "gmres", "sgs", "ilu", "serve"])
    f32 = rng.random() < 0.3 if do in ("spmv", "smooth", "blas1", "sgs", "ilu", "cg") else False
    three = rng.random() < 0.6
    c = {"do": do, "op": "none", "nx": 1, "ny": 1, "nz": 1, "f32": f32}
    if do == "blas1":
        c["nx"] = _size(rng, 1000, 4_000_000)
        return c
    if do == "serve":
        return {"do": do, "op": "fv", "nmin": 1000, "nmax": _size(rng, 10_000, 300_000), "count": rng.randint(4, 32),
                "mix": rng.randint(0, 10_000), "f32": False}
    lo, hi = {"spmv": (1000, 6_000_000), "smooth": (1000, 3_000_000), "cg": (1000, 1_800_000),
              "cgmc": (4000, 2_500_000), "dc": (4000, 5_000_000), "gmres": (4000, 1_500_000),
              "sgs": (1000, 1_500_000), "ilu": (1000, 1_500_000)}[do]
    n = _size(rng, lo, hi)
    if do in ("gmres", "ilu"):
        c["op"] = "upwind"
    elif do in ("cgmc", "dc", "sgs"):
        c["op"] = "fv"
    else:
        c["op"] = rng.choice(["q1", "fv"])
        if c["op"] == "q1":
            c["op"] = "q1_3d" if three else "q1_2d"
            if three:
                n = min(n, 2_000_000)
    if not three:
        # the 2D systems need more iterations for the same number of unknowns
        n = min(n, {"cg": 300_000, "cgmc": 300_000, "dc": 300_000, "gmres": 30_000}.get(do, n))
    c["nx"], c["ny"], c["nz"] = _shape(rng, n, three)
    return c


# -------------------------------------------------------------- the operators

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed, stream):
    g = torch.Generator(device="cpu")
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _uniform(n, seed, stream):
    """n values in [-1, 1) on the device."""
    return (torch.rand(n, generator=_gen(seed, stream), dtype=torch.float64) * 2 - 1).to(_dev())


def _cells(n, sigma, seed):
    """Lognormal cell coefficients."""
    return torch.exp(sigma * torch.randn(n, generator=_gen(seed, 1), dtype=torch.float64))


def _grid(nx, ny, nz):
    d = _dev()
    i = torch.arange(nx * ny * nz, device=d)
    return i % nx, (i // nx) % ny, i // (nx * ny)


def _stencil(op, nx, ny, nz, kc):
    """(offsets ascending, coefficients [K, n], present [K, n]) of an operator."""
    X, Y, Z = _grid(nx, ny, nz)
    n, d = nx * ny * nz, _dev()

    def there(dx, dy, dz):
        return ((X + dx >= 0) & (X + dx < nx) & (Y + dy >= 0) & (Y + dy < ny) & (Z + dz >= 0) & (Z + dz < nz))

    offs, coef, have = [], [], []
    if op in ("q1_2d", "q1_3d"):
        h = 1.0 / (nx + 1)
        for dz in ((-1, 0, 1) if op == "q1_3d" else (0,)):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    k = abs(dx) + abs(dy) + abs(dz)
                    v = (8.0 * h / 3.0, 0.0, -h / 6.0, -h / 12.0)[k] if op == "q1_3d" else (8.0 / 3.0, -1.0 / 3.0, -1.0 / 3.0)[k]
                    m = there(dx, dy, dz)
                    offs.append(dx + nx * (dy + ny * dz))
                    coef.append(torch.where(m, torch.full((n,), v, dtype=torch.float64, device=d), 0.0))
                    have.append(m)
        return offs, torch.stack(coef), torch.stack(have)
    axes = [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
    if nz == 1:
        axes = axes[1:5]
    diag = torch.zeros(n, dtype=torch.float64, device=d)
    if op == "upwind":
        h, eps, peclet = 1.0 / nx, 1e-2, 5.0
        s = peclet * eps / (h * math.sqrt(0.59))
        vel = (-s * ((Y.double() + 0.5) * h - 0.5), s * ((X.double() + 0.5) * h - 0.5),
               torch.full((n,), 0.3 * s, dtype=torch.float64, device=d))
    side = {}
    for a in axes:
        m = there(*a)
        o = a[0] + nx * (a[1] + ny * a[2])
        if op == "fv":
            other = kc[(torch.arange(n, device=d) + o).clamp(0, n - 1)]
            t = torch.where(m, 2.0 * kc * other / (kc + other), 0.0)
            c = -t
            diag = diag + torch.where(m, t, 2.0 * kc)
        else:
            axis = [abs(v) for v in a].index(1)
            vh = vel[axis] * h * -sum(a)      # positive: the flow comes from this neighbour
            c = torch.where(m, -eps - vh.clamp(min=0.0), 0.0)
            diag = diag + torch.where(m, eps, 2.0 * eps) + vh.clamp(min=0.0)
        side[o] = (c, m)
    side[0] = (diag, torch.ones(n, dtype=torch.bool, device=d))
    offs = sorted(side)
    return offs, torch.stack([side[o][0] for o in offs]), torch.stack([side[o][1] for o in offs])


def _csr(st):
    """Host CSR arrays of a stencil operator."""
    offs, coef, have = st
    n = coef.shape[1]
    hT = have.t().contiguous()
    col = (torch.arange(n, device=coef.device)[:, None] + torch.tensor(offs, device=coef.device)[None, :])[hT]
    val = coef.t().contiguous()[hT]
    row = torch.zeros(n + 1, dtype=torch.int64, device=coef.device)
    row[1:] = torch.cumsum(hT.sum(1), 0)
    return row.to(torch.int32).cpu().numpy(), col.to(torch.int32).cpu().numpy(), val.cpu().numpy()


def _operator(case, seed):
    n = case["nx"] * case["ny"] * case["nz"]
    kc = _cells(n, 1.0, seed).to(_dev()) if case["op"] == "fv" else None
    return _stencil(case["op"], case["nx"], case["ny"], case["nz"], kc)


def _serve_shapes(case):
    """Sizes of a serving mix: log-uniform from nmin to nmax unknowns, half 2D, half 3D."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["count"]):
        n = math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))
        if rng.random() < 0.5:
            s = max(2, int(round(n ** (1.0 / 3.0))))
            out.append((s, s, s))
        else:
            s = max(2, int(round(n ** 0.5)))
            out.append((s, s, 1))
    return out


def _parity_order(case):
    """Rows by colour of the 5- / 7-point grid: first-fit colouring is the parity of x + y + z."""
    X, Y, Z = _grid(case["nx"], case["ny"], case["nz"])
    p = (X + Y + Z) % 2
    return torch.cat([torch.nonzero(p == 0)[:, 0], torch.nonzero(p == 1)[:, 0]])


# ------------------------------------------------------------ prepare and run

class _Shared:
    """A device vector's memory as seen by torch (keeps the vector alive)."""

    def __init__(self, v):
        self.vector = v
        self.__cuda_array_interface__ = {"shape": (v.n,), "typestr": "<f4" if v.dtype == np.float32 else "<f8",
                                         "data": (v.device_ptr(), False), "version": 2, "strides": None}


def _tensor(v):
    return torch.as_tensor(_Shared(v), device="cuda")


def prepare(case, seed):
    P, ctx = _pkg(), _context()
    dt = np.float32 if case["f32"] else np.float64
    do = case["do"]
    s = {"P": P, "case": dict(case)}
    if do == "blas1":
        for k, name in enumerate(("x", "r", "p", "q")):
            s[name] = P.Vector(ctx, _uniform(case["nx"], seed, 10 + k).cpu().numpy().astype(dt), dt)
            s["t" + name] = _tensor(s[name])
        return s
    if do == "serve":
        s["jobs"] = []
        for k, (nx, ny, nz) in enumerate(_serve_shapes(case)):
            n = nx * ny * nz
            s["jobs"].append((nx, ny, nz, _cells(n, 0.5, seed * 64 + k).numpy(),
                              _uniform(n, seed * 64 + k, 2).cpu().numpy()))
        s["engine"] = P.BatchEngine(ctx, max_systems=64, hbm_budget=1 << 31, chunk=16, rtol=1e-10, atol=0.0,
                                    outer_maxits=30, inner_rtol=1e-4, inner_maxits=20000)
        return s
    st = _operator(case, seed)
    row, col, val = _csr(st)
    n = len(row) - 1
    b = _uniform(n, seed, 2)
    if do in ("cgmc", "dc"):
        A0 = P.CsrMatrix(ctx, row, col, val)
        nc, _, sizes, perm = A0.multicoloring()
        A = A0.permuted(perm)
        b = b.cpu().numpy()[perm]
        s["A"] = A
        if do == "cgmc":
            s["M"] = P.Preconditioner.mcsgs(A, sizes, 1.0)
        else:
            s["A32"] = P.CsrMatrix.cast_of(A, np.float32)
            s["M"] = P.Preconditioner.mcsgs(s["A32"], sizes, 1.0)
            s["atol"] = 1e-10 * float(np.linalg.norm(b))
    else:
        b = b.cpu().numpy().astype(dt)
        if do == "ilu" or do == "gmres":
            lu = P.ilu0_factor(row, col, val)
            s["LU"] = P.CsrMatrix(ctx, row, col, lu.astype(dt))
            s["M"] = P.Preconditioner.ilu0(s["LU"], row, col)
        if do != "ilu":
            s["A"] = P.CsrMatrix(ctx, row, col, val.astype(dt))
        if do == "cg":
            s["M"] = P.Preconditioner.jacobi(s["A"])
        if do == "sgs":
            s["M"] = P.Preconditioner.sgs(s["A"], row, col)
        if do == "smooth":
            s["A"].swap_diag_front()
    s["b"] = P.Vector(ctx, b, dt)
    s["x"] = P.Vector(ctx, n, dt)
    s["tx"] = _tensor(s["x"])
    return s


def run(s):
    P, do = s["P"], s["case"]["do"]
    if do == "blas1":
        pq = s["p"].dot(s["q"])
        s["x"].axpy(s["p"], 1e-3)
        s["r"].axpy(s["q"], -1e-3)
        rr = s["r"].nrm2()
        s["p"].scaleadd(0.5, s["r"])
        return [pq, rr, s["tx"], s["tr"], s["tp"]]
    if do == "serve":
        E, todo, at, out = s["engine"], list(range(len(s["jobs"]))), {}, [None] * len(s["jobs"])
        left = len(todo)
        while left:
            while todo:
                nx, ny, nz, k, b = s["jobs"][todo[0]]
                rid = E.submit_fv(nx, ny, nz, k, b)
                if rid is None:
                    break
                at[rid] = todo.pop(0)
            E.step()
            for rid in E.finished():
                j = at.pop(rid)
                out[j], _ = E.collect(rid, len(s["jobs"][j][4]))
                left -= 1
        return out
    if do == "spmv":
        s["A"].spmv(s["b"], s["x"])
    elif do in ("sgs", "ilu"):
        s["M"].apply(s["b"], s["x"])
    else:
        s["x"].zeros()
        if do == "smooth":
            P.jacobi(s["A"], s["b"], s["x"], mode=P.JACOBI_SMOOTH_DAMPED, w=0.8, inner_iter=1, smooth_iter=3)
        elif do == "cg":
            # single precision: a tolerance its residuals can reach
            P.pcg(s["A"], s["b"], s["x"], s["M"], maxits=20000, atol=0.0, rtol=1e-4 if s["case"]["f32"] else 1e-8)
        elif do == "cgmc":
            P.pcg(s["A"], s["b"], s["x"], s["M"], maxits=20000, atol=0.0, rtol=1e-10)
        elif do == "dc":
            P.dc(s["A"], s["A32"], s["b"], s["x"], s["M"], outer=(60, s["atol"], 0.0, 1e10),
                 inner=(20000, s["atol"], 1e-2, 1e10), keep_direction=True)
        else:
            P.gmres(s["A"], s["b"], s["x"], s["M"], m=30, maxits=20000, atol=0.0, rtol=1e-8)
    return [s["tx"]]


# -------------------------------------------------------------- compulsory work

def _counts(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    if case["op"] == "q1_3d":
        return n, (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    if case["op"] == "q1_2d":
        return n, (3 * nx - 2) * (3 * ny - 2)
    nnz = n + 2 * ((nx - 1) * ny * nz + nx * (ny - 1) * nz)
    return n, nnz + (2 * nx * ny * (nz - 1) if nz > 1 else 0)


def _steps(do, side, three):
    """Iterations of the solves, about: they grow with the longest side."""
    if do == "cg":
        return (2.2 if not three else 2.0) * side + 10
    if do in ("cgmc", "dc"):
        return (3.0 if not three else 2.3) * side + 10
    if do == "serve":
        return 3.5 * side + 10
    return 1.5 * side + 5


def work(case):
    do, v = case["do"], 4 if case["f32"] else 8
    if do == "blas1":
        # five operations: 2 + 3 + 3 + 1 + 3 vectors
        return {"bytes": 12 * v * case["nx"], "flops": 10 * case["nx"]}
    if do == "serve":
        by = fl = 0.0
        for nx, ny, nz in _serve_shapes(case):
            n, nnz = _counts({"nx": nx, "ny": ny, "nz": nz, "op": "fv"})
            it = _steps("serve", nx, nz > 1)
            by += it * (8 * nnz + 60 * n)
            fl += it * (2 * nnz + 14 * n)
        return {"bytes": by, "flops": fl}
    n, nnz = _counts(case)
    it = _steps(do, max(case["nx"], case["ny"], case["nz"]), case["nz"] > 1)
    spmv = (v + 4) * nnz + (2 * v + 4) * n
    if do == "spmv":
        return {"bytes": spmv, "flops": 2 * nnz}
    if do == "smooth":
        return {"bytes": 3 * ((v + 4) * nnz + (4 * v + 4) * n), "flops": 3 * (2 * nnz + 4 * n)}
    if do in ("sgs", "ilu"):
        return {"bytes": (v + 4) * nnz + 4 * v * n, "flops": 2 * nnz + 2 * n}
    if do == "cg":
        return {"bytes": it * ((v + 4) * nnz + 12.5 * v * n), "flops": it * (2 * nnz + 12 * n)}
    if do == "cgmc":
        return {"bytes": it * (24 * nnz + 150 * n), "flops": it * (4 * nnz + 16 * n)}
    if do == "dc":
        return {"bytes": it * (16 * nnz + 76 * n), "flops": it * (4 * nnz + 16 * n)}
    # gmres: SpMV, the ILU(0) apply, the basis read once per orthogonalisation
    # (15.5 vectors on average) and a new vector written
    return {"bytes": it * (24 * nnz + 44 * n + 8 * n * 17.5), "flops": it * (4 * nnz + 66 * n)}


def tolerance(case):
    do = case["do"]
    if do in ("spmv", "smooth", "sgs", "ilu"):
        # sums of a few terms; the sweeps carry a rounding along their rows
        return {"rel": 4e-7, "max": 2e-5} if case["f32"] else {"rel": 1e-14, "max": 1e-12}
    if do == "blas1":
        return {"rel": 4e-7, "max": 2e-5} if case["f32"] else {"rel": 1e-13, "max": 1e-12}
    # solves stop at a residual, so their results are as far apart as one
    # step's error at that residual
    return {"rel": 1e-3, "max": 4e-2} if case["f32"] else {"rel": 1e-6, "max": 4e-5}


# --------------------------------------------------------- the result in 64 bits

def _apply(st, x, only=None):
    """A x of a stencil operator; `only` selects offsets."""
    offs, coef, _ = st
    m = max(abs(o) for o in offs)
    xp = torch.nn.functional.pad(x, (m, m))
    y = torch.zeros_like(x)
    for k, o in enumerate(offs):
        if only is None or only(o):
            y.addcmul_(coef[k], xp[m + o:m + o + x.numel()])
    return y


def _solve_spd(st, b, tol=1e-14, most=20000):
    inv = 1.0 / st[1][st[0].index(0)]
    x, r = torch.zeros_like(b), b.clone()
    z = inv * r
    p, rz, stop = z.clone(), torch.dot(r, z), tol * float(b.norm())
    for it in range(most):
        if it % 20 == 0 and float(r.norm()) <= stop:
            break
        q = _apply(st, p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        z = inv * r
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _solve_general(st, b, tol=1e-13, most=5000):
    """BiCGSTAB with Jacobi scaling, restarted from the true residual."""
    inv = 1.0 / st[1][st[0].index(0)]
    x, nb = torch.zeros_like(b), float(b.norm())
    for _ in range(6):
        r = b - _apply(st, x)
        if float(r.norm()) <= tol * nb:
            break
        r0, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
        rho = al = om = torch.ones((), dtype=torch.float64, device=b.device)
        start = float(r.norm())
        for it in range(most):
            new = torch.dot(r0, r)
            p = r + (new / rho) * (al / om) * (p - om * v)
            rho = new
            ph = inv * p
            v = _apply(st, ph)
            al = rho / torch.dot(r0, v)
            sv = r - al * v
            sh = inv * sv
            t = _apply(st, sh)
            om = torch.dot(t, sv) / torch.dot(t, t)
            x += al * ph + om * sh
            r = sv - om * t
            if it % 20 == 19:
                now = float(r.norm())
                if now <= tol * nb or now <= 1e-12 * start or now > 1e3 * start:
                    break
    return x


def _levels(case):
    X, Y, Z = _grid(case["nx"], case["ny"], case["nz"])
    key, order = torch.sort(X + Y + Z, stable=True)
    return list(torch.split(order, torch.bincount(key).tolist()))


def _sweeps(case, st, b, ilu):
    """ILU(0) or symmetric Gauss-Seidel apply by levels of x + y + z."""
    offs, coef, have = st
    k0 = offs.index(0)
    n, m = coef.shape[1], max(abs(o) for o in offs)
    rows = _levels(case)
    lo = [k for k, o in enumerate(offs) if o < 0]
    up = [k for k, o in enumerate(offs) if o > 0]
    d, L = coef[k0].clone(), {k: coef[k].clone() for k in lo}
    if ilu:
        # a 5- / 7-point pattern has no fill: only the diagonal changes
        for r in rows:
            for k in lo:
                j = (r + offs[k]).clamp(0, n - 1)
                l = torch.where(have[k][r], coef[k][r] / d[j], 0.0)
                L[k][r] = l
                d[r] -= torch.where(have[k][r], l * coef[offs.index(-offs[k])][j], 0.0)
    y = torch.zeros(n + 2 * m, dtype=torch.float64, device=b.device)
    for r in rows:
        t = b[r].clone()
        for k in lo:
            t -= L[k][r] * y[m + r + offs[k]]
        y[m + r] = t if ilu else t / d[r]
    z = torch.zeros_like(y)
    for r in reversed(rows):
        t = y[m + r] if ilu else y[m + r] * d[r]
        for k in up:
            t = t - coef[k][r] * z[m + r + offs[k]]
        z[m + r] = t / d[r]
    return z[m:m + n]


def exact(case, seed):
    do, f32 = case["do"], case["f32"]

    def rounded(t):
        return t.float().double() if f32 else t

    if do == "blas1":
        x, r, p, q = (rounded(_uniform(case["nx"], seed, 10 + k)) for k in range(4))
        small = float(np.float32(1e-3)) if f32 else 1e-3
        pq = float(torch.dot(p, q))
        x = x + small * p
        r = r - small * q
        return [pq, float(r.norm()), x, r, 0.5 * p + r]
    if do == "serve":
        out = []
        for k, (nx, ny, nz) in enumerate(_serve_shapes(case)):
            n = nx * ny * nz
            st = _stencil("fv", nx, ny, nz, _cells(n, 0.5, seed * 64 + k).to(_dev()))
            out.append(_solve_spd(st, _uniform(n, seed * 64 + k, 2)).cpu().numpy())
        return out
    st = _operator(case, seed)
    n = st[1].shape[1]
    b = rounded(_uniform(n, seed, 2))
    if do == "ilu" and f32:
        return None   # the factors are rounded after the factorisation
    st = (st[0], rounded(st[1]), st[2])
    if do == "spmv":
        return [_apply(st, b)]
    if do in ("sgs", "ilu"):
        return [_sweeps(case, st, b, do == "ilu")]
    if do == "smooth":
        d = st[1][st[0].index(0)]
        w = float(np.float32(0.8)) if f32 else 0.8
        x = torch.zeros_like(b)
        for _ in range(3):
            x = (1.0 - w) * x + w * (b - _apply(st, x, lambda o: o != 0)) / d
        return [x]
    if do == "gmres":
        return [_solve_general(st, b)]
    x = _solve_spd(st, b)
    if do in ("cgmc", "dc"):
        x = x[_parity_order(case)]
    return [x]
