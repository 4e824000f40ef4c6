"""Performance cases of f3r_amd: what a program that uses this framework has it
do, through the public Python entry points.

Every case is a dict of plain values.  `listed()` gives the fixed ones,
`draw(rng)` one more of the same ranges, `prepare(case, seed)` what a program
holds before the call (matrix handles, preconditioner, solver, device
vectors), `run(state)` one pass, `work(case)` the bytes and operations the
path cannot do without, and `exact(case, seed)` the same outputs in 64 bits
from plain torch.

Kinds of case:
  solve  F3R(...).solve(b, x) to 1e-8: the framework's main path
  nest   a nest composed of FGMRES levels over a preconditioner applied directly
  batch  many systems with several right-hand sides each, solved in lockstep
  spmv   one product or residual with a SELL or CSR matrix
  cg     a Krylov loop that a program writes itself from the vector operations
  learn  loss and gradient of the learned preconditioner over one system
Matrices (all scaled by algorithm.scaling before use, as the solver's users do):
  27c    27-point, constant coefficients, nonsymmetric along x (HPCG's pattern)
  7v     7-point lognormal diffusion, upwind convection for peclet > 0
  27v    27-point, lognormal coefficients (a trilinear element mesh)
  dom    7- or 27-point, unit off-diagonals, random dominance margin
  graph  rows of uneven length, mostly near the diagonal (circuits, meshes)
"""
import ctypes
import math

import torch

import f3r_amd as F
from f3r_amd import learn

EPS = 1e-8
NEST = (100, 8, 4, 2)   # m1, m2, m3, m4 of the reference's driver
STEPS = 4               # outer steps counted as necessary in work(); solves here take 2 to 8
_BYTES = {"f64": 8, "f32": 4, "f16": 2}
_TORCH = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16}


# ------------------------------------------------------------------ cases ---
def listed():
    return [
        # the reference's headline workload at its stated size: the bench of this repository
        {"name": "solve_27c_128", "kind": "solve", "matrix": "27c", "nx": 128, "ny": 128, "nz": 128,
         "precond": "sdainv", "variant": "half"},
        # variable coefficients at the size the learned family and the precision study use
        {"name": "solve_7v_96", "kind": "solve", "matrix": "7v", "nx": 96, "ny": 96, "nz": 96, "peclet": 0.0,
         "precond": "sdainv", "variant": "half"},
        # a trilinear element mesh with ragged edges: 27 different values in every row
        {"name": "solve_27v_ragged", "kind": "solve", "matrix": "27v", "nx": 75, "ny": 70, "nz": 67,
         "precond": "sdainv", "variant": "half"},
        # a small system, as in a time-stepping loop: bound by latency and launches
        {"name": "solve_27c_small", "kind": "solve", "matrix": "27c", "nx": 25, "ny": 24, "nz": 23,
         "precond": "sdainv", "variant": "half"},
        # convection-diffusion with the reference's CPU-path preconditioner, block-Jacobi ILU(0) of 112 blocks
        {"name": "solve_7v_bjilu", "kind": "solve", "matrix": "7v", "nx": 64, "ny": 64, "nz": 64, "peclet": 10.0,
         "precond": "bjilu0", "variant": "half"},
        # the reference driver's FLOAT build (no fp16 anywhere)
        {"name": "solve_27c_float", "kind": "solve", "matrix": "27c", "nx": 65, "ny": 64, "nz": 63,
         "precond": "sdainv", "variant": "float"},
        # F3 of the reference's depth study, composed from FGMRES objects
        {"name": "nest_7v_48", "kind": "nest", "matrix": "7v", "nx": 48, "ny": 50, "nz": 49, "peclet": 10.0},
        # the batched configuration (sizes 16^3..64^3, half 7-point, half 27-point, 4 right-hand sides each)
        {"name": "batch_16x4", "kind": "batch", "systems": 16, "rhs": 4, "lo": 16, "hi": 64, "gseed": 1},
        # single products: an fp16 SELL product, and the fp64 residual of an outer iteration
        {"name": "spmv_sell_f16", "kind": "spmv", "matrix": "27v", "nx": 100, "ny": 96, "nz": 97, "format": "sell",
         "dtype": "f16", "op": "operate"},
        # CSR rows of uneven length
        {"name": "spmv_csr_f64_graph", "kind": "spmv", "matrix": "graph", "n": 300007, "mean": 14, "format": "csr",
         "dtype": "f64", "op": "residual"},
        # a program's own CG loop over the vector operations: short calls, a host scalar each
        {"name": "cg_7v_small", "kind": "cg", "matrix": "7v", "nx": 24, "ny": 23, "nz": 25, "peclet": 0.0, "steps": 8},
        # a training step's loss and gradient
        {"name": "learn_64", "kind": "learn", "nx": 64, "probes": 8, "loss": 0},
    ]


def _edges(rng, lo, hi):
    """three grid edges whose volume is spread over its logarithm"""
    e = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(lo, min(hi, int(round(e * rng.uniform(0.9, 1.1))))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "nest", "batch", "spmv", "spmv", "cg", "learn"])
    if kind == "solve":
        variant = rng.choice(["half", "half", "half", "float", "double"])
        precond = rng.choice(["sdainv", "sdainv", "bjilu0"])
        matrix = rng.choice(["27c", "7v", "27v"]) if precond == "sdainv" else "7v"
        hi = 128 if matrix != "27v" and precond == "sdainv" and variant == "half" else 80
        if precond == "bjilu0":
            hi = 56
        nx, ny, nz = _edges(rng, 16, hi)
        c = {"kind": "solve", "matrix": matrix, "nx": nx, "ny": ny, "nz": nz, "precond": precond, "variant": variant}
        if matrix == "7v":
            c["peclet"] = rng.choice([0.0, 10.0])
        return c
    if kind == "nest":
        nx, ny, nz = _edges(rng, 16, 64)
        return {"kind": "nest", "matrix": "7v", "nx": nx, "ny": ny, "nz": nz, "peclet": rng.choice([0.0, 10.0])}
    if kind == "batch":
        lo = rng.choice([16, 20, 24])
        return {"kind": "batch", "systems": rng.randint(2, 16), "rhs": rng.choice([1, 2, 4]), "lo": lo,
                "hi": rng.randint(lo + 8, 60), "gseed": rng.randint(2, 1 << 20)}
    if kind == "spmv":
        fmt, dt, op = rng.choice(["sell", "csr"]), rng.choice(["f64", "f32", "f16"]), rng.choice(["operate", "residual"])
        if rng.random() < 0.4:
            return {"kind": "spmv", "matrix": "graph", "n": int(math.exp(rng.uniform(math.log(5e3), math.log(5e5)))),
                    "mean": rng.randint(6, 24), "format": fmt, "dtype": dt, "op": op}
        nx, ny, nz = _edges(rng, 16, 100)
        return {"kind": "spmv", "matrix": rng.choice(["27c", "27v", "7v"]), "nx": nx, "ny": ny, "nz": nz, "peclet": 0.0,
                "format": fmt, "dtype": dt, "op": op}
    if kind == "cg":
        nx, ny, nz = _edges(rng, 16, 80)
        return {"kind": "cg", "matrix": "7v", "nx": nx, "ny": ny, "nz": nz, "peclet": 0.0, "steps": rng.randint(4, 12)}
    return {"kind": "learn", "nx": rng.randint(20, 64), "probes": rng.choice([2, 4, 8]), "loss": rng.choice([0, 1])}


# --------------------------------------------------------------- matrices ---
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _gaussian(nx, ny, nz, corr, seed):
    """unit-variance Gaussian field: white noise smoothed along each axis"""
    g = torch.randn((1, 1, nz, ny, nx), dtype=torch.float64, device=_device(), generator=_generator(seed))
    r = int(math.ceil(2 * corr))
    w = torch.exp(-0.5 * (torch.arange(-r, r + 1, dtype=torch.float64, device=g.device) / corr) ** 2)
    g = g[0, 0]
    for axis in range(3):
        out = torch.zeros_like(g)
        m = g.shape[axis]
        for k in range(-r, r + 1):
            a, b = max(0, -k), min(m, m - k)
            if a < b:
                out.narrow(axis, a, b - a).add_(g.narrow(axis, a + k, b - a), alpha=float(w[k + r]))
        g = out
    return ((g - g.mean()) / g.std()).reshape(-1)


def _grid(case, seed):
    """(columns, values) of a grid matrix, one row per unknown, -1 where there is no entry"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dev = _device()
    n = nx * ny * nz
    row = torch.arange(n, device=dev, dtype=torch.int32)
    i, j, k = row % nx, (row // nx) % ny, row // (nx * ny)
    m = case["matrix"]
    npts = case.get("npts", 7 if m == "7v" else 27)
    kap = None
    if m in ("7v", "27v"):
        rng = torch.Generator().manual_seed(int(seed) * 2 + 1)
        sig, corr = (0.5 + 1.0 * torch.rand(1, generator=rng).item(), 2.0 + 6.0 * torch.rand(1, generator=rng).item())
        kap = torch.exp(sig * _gaussian(nx, ny, nz, corr, seed))
    cols, vals, centre = [], [], None
    diag = torch.zeros(n, dtype=torch.float64, device=dev)
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                man = abs(dx) + abs(dy) + abs(dz)
                if npts == 7 and man > 1:
                    continue
                if man == 0:
                    centre = len(cols)
                    cols.append(row.clone())
                    vals.append(None)
                    continue
                ok = (i + dx >= 0) & (i + dx < nx) & (j + dy >= 0) & (j + dy < ny) & (k + dz >= 0) & (k + dz < nz)
                c = row + ((dz * ny + dy) * nx + dx)
                if kap is not None:
                    o = kap[c.clamp(0, n - 1).long()]
                    v = 2 * kap * o / (kap + o)
                    # Dirichlet boundary: the missing neighbour's share stays on the diagonal
                    diag += torch.where(ok, v, 2 * kap if m == "7v" else kap)
                    v = -v
                    if m == "7v" and dx == -1:
                        v = v - case["peclet"]   # first-order upwind convection along +x
                elif m == "27c":
                    v = torch.full((n,), -1.0 + 0.5 * (dx > 0) - 0.5 * (dx < 0), dtype=torch.float64, device=dev)
                else:
                    v = torch.full((n,), -1.0, dtype=torch.float64, device=dev)
                    diag += ok
                cols.append(torch.where(ok, c, torch.full_like(c, -1)))
                vals.append(torch.where(ok, v, torch.zeros_like(v)))
    if m == "27c":
        diag.fill_(26.0)
    elif m == "dom":
        diag *= 1.0 + case["margin"]
    else:
        diag += case.get("peclet", 0.0)
    vals[centre] = diag
    return torch.stack(cols, 1), torch.stack(vals, 1)


def _graph(case, seed):
    """(rows, columns, values), sorted: uneven rows, most entries near the diagonal, a diagonal in every row"""
    n, dev, g = case["n"], _device(), _generator(seed)
    u = torch.rand(n, dtype=torch.float64, device=dev, generator=g)
    ln = (0.5 * case["mean"] / (1 - u).clamp_min(1e-3) ** 0.5).round().long().clamp(1, 200)   # a heavy tail
    row = torch.repeat_interleave(torch.arange(n, device=dev), ln)
    near = torch.randint(-200, 201, row.shape, device=dev, generator=g) + row
    far = torch.randint(0, n, row.shape, device=dev, generator=g)
    col = torch.where(torch.rand(row.shape, device=dev, generator=g) < 0.9, near.clamp(0, n - 1), far)
    key = torch.unique(torch.cat([row * n + col, torch.arange(n, device=dev) * (n + 1)]))
    row, col = key // n, key % n
    val = torch.rand(row.shape, dtype=torch.float64, device=dev, generator=g) * 2 - 1
    off = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, row, torch.where(row == col, 0.0, val.abs()))
    return row, col, torch.where(row == col, 1.5 * (off[row] + 1.0), val)


def _csr(case, seed):
    """host CSR of the case's matrix, scaled"""
    if case["matrix"] == "graph":
        row, col, val = _graph(case, seed)
        n, cnt = case["n"], torch.bincount(row, minlength=case["n"])
    else:
        c, v = _grid(case, seed)
        n, on = c.shape[0], c >= 0
        cnt, col, val = on.sum(1), c[on], v[on]
    rptr = torch.zeros(n + 1, dtype=torch.int32)
    rptr[1:] = torch.cumsum(cnt, 0).to(torch.int32).cpu()
    A = F.CSR(n, rptr.numpy(), col.to(torch.int32).cpu().numpy(), val.cpu().numpy())
    return F.algorithm.scaling(A)


def _matvec(case, seed):
    """(n, x -> A x in 64 bits) of the scaled matrix, from plain torch"""
    if case["matrix"] == "graph":
        row, col, val = _graph(case, seed)
        n = case["n"]
        d = torch.zeros(n, dtype=torch.float64, device=val.device)
        d[row[row == col]] = val[row == col].abs().sqrt()
        val = val / (d[row] * d[col])
        return n, lambda x: torch.zeros_like(x).index_add_(0, row, val * x[col])
    c, v = _grid(case, seed)
    n = c.shape[0]
    at = c.clamp_min(0).long()
    d = v.gather(1, (c == torch.arange(n, device=c.device, dtype=torch.int32)[:, None]).int().argmax(1, True)).abs().sqrt()
    v = torch.where(c >= 0, v / (d * d[:, 0][at]), torch.zeros_like(v))
    return n, lambda x: (v * x[at]).sum(1)


def _solve64(n, A, b):
    """A x = b in 64 bits: BiCGSTAB, restarted on its true residual"""
    x = torch.zeros_like(b)
    best = None
    for _ in range(6):
        r = b - A(x)
        rel = float(r.norm() / b.norm())
        if best is None or rel < best[0]:
            best = (rel, x.clone())
        if rel < 1e-13:
            break
        rh, p = r.clone(), r.clone()
        rho = torch.dot(rh, r)
        d = torch.zeros_like(b)
        stop = max(1e-14 * float(b.norm()), 1e-9 * float(r.norm()))
        for it in range(1500):
            v = A(p)
            al = rho / torch.dot(rh, v)
            s = r - al * v
            t = A(s)
            om = torch.dot(t, s) / torch.dot(t, t)
            d += al * p + om * s
            r = s - om * t
            if it % 8 == 7 and not float(r.norm()) > stop:
                break
            rho1 = torch.dot(rh, r)
            p = r + (rho1 / rho) * (al / om) * (p - om * v)
            rho = rho1
        if bool(torch.isfinite(d).all()):
            x = x + d
    return best[1] if best[0] < 1e-11 else None


# ---------------------------------------------------------------- vectors ---
_CTX = []


def _ctx():
    """the program's one context"""
    if not _CTX:
        _CTX.append(F.Context(0))
    return _CTX[0]


class _Memory:
    """the device memory of an f3r_amd vector, for torch.as_tensor (which holds this object, and so the vector)"""

    def __init__(self, v, typestr):
        self.v = v
        p = ctypes.c_void_p()
        F.check(F.lib.f3r_vec_info(v.handle, None, None, ctypes.byref(p)), "vec_info")
        self.__cuda_array_interface__ = {"shape": (v.n,), "typestr": typestr, "data": (p.value, False), "version": 2}


def _tensor(v, dtype):
    return torch.as_tensor(_Memory(v, {"f64": "<f8", "f32": "<f4", "f16": "<f2"}[dtype]), device="cuda")


def _uniform(n, seed, salt):
    """n values in [-1, 1], on the device"""
    return torch.rand(n, dtype=torch.float64, device=_device(), generator=_generator((int(seed) << 8) + salt)) * 2 - 1


def _vector(t, dtype="f64"):
    return F.vector.from_numpy(_ctx(), t.to(_TORCH[dtype]).cpu().numpy(), dtype)


# ---------------------------------------------------------------- prepare ---
def _precond(case, A, dtype):
    if case["precond"] == "bjilu0":
        return F.ILU0(A, 112, 1.0, dtype, ctx=_ctx(), device=True)
    return F.SDAINV(A, 0.1, 1.0, dtype, ctx=_ctx(), device=True)


def _family(case):
    """[(points, edge, dominance margin)] of a batch"""
    g = torch.Generator().manual_seed(case["gseed"])
    u = torch.rand(2 * case["systems"], dtype=torch.float64, generator=g).tolist()
    span = case["hi"] - case["lo"] + 1
    return [(7 if s % 2 == 0 else 27, case["lo"] + int(u[2 * s] * span), 0.5 + 1.5 * u[2 * s + 1])
            for s in range(case["systems"])]


def _batch_matrix(points, edge, margin):
    return {"matrix": "dom", "npts": points, "nx": edge, "ny": edge, "nz": edge, "margin": margin}


def prepare(case, seed):
    return {"solve": _prepare_solve, "nest": _prepare_nest, "batch": _prepare_batch, "spmv": _prepare_spmv,
            "cg": _prepare_cg, "learn": _prepare_learn}[case["kind"]](case, seed)


def _prepare_solve(case, seed):
    ctx, A = _ctx(), _csr(case, seed)
    dt = {"half": "f16", "float": "f32", "double": "f64"}[case["variant"]]
    M = _precond(case, A, dt)
    S = F.F3R(ctx, A, M, m=NEST, variant=case["variant"], eps=EPS, device_build=True)
    b, x = _vector(_uniform(A.n, seed, 1)), F.vector(ctx, "f64", A.n)
    return {"run": _run_solve, "A": A, "M": M, "S": S, "b": b, "x": x, "out": _tensor(x, "f64")}


def _prepare_nest(case, seed):
    ctx, A = _ctx(), _csr(case, seed)
    M = F.SDAINV(A, 0.1, 1.0, "f16", ctx=ctx, device=True)
    S = F.Restarted(ctx, A, F.FGMRES("f64", F.FGMRES("f32", F.FGMRES("f16", M, 8), 8), 100, normalize=True, T="f64"),
                    20, eps=EPS)
    b, x = _vector(_uniform(A.n, seed, 1)), F.vector(ctx, "f64", A.n)
    return {"run": _run_solve, "A": A, "M": M, "S": S, "b": b, "x": x, "out": _tensor(x, "f64")}


def _prepare_batch(case, seed):
    ctx = _ctx()
    As, Ps, rows = [], [], []
    for points, edge, margin in _family(case):
        A = _csr(_batch_matrix(points, edge, margin), seed)
        P = F.SDAINV(A, 0.1, 1.0, "f16", ctx=ctx, device=True)
        As += [A] * case["rhs"]
        Ps += [P] * case["rhs"]
        rows += [A.n] * case["rhs"]
    total = sum(rows)
    b, x = _vector(_uniform(total, seed, 1)), F.vector(ctx, "f64", total)
    at = [sum(rows[:s]) for s in range(len(rows))]
    return {"run": _run_batch, "keep": (As, Ps), "B": F.Batch(ctx, As, Ps, m=NEST, eps=EPS), "b": b, "x": x,
            "bs": [b.view(o, n) for o, n in zip(at, rows)], "xs": [x.view(o, n) for o, n in zip(at, rows)],
            "out": _tensor(x, "f64")}


def _prepare_spmv(case, seed):
    ctx, A, dt = _ctx(), _csr(case, seed), case["dtype"]
    if case["format"] == "csr":
        S = F.CSRDevice(ctx, A, dt)
    else:   # stencils in the chunk-offset layout, uneven rows sorted in windows
        grid = case["matrix"] != "graph"
        S = F.SELL(ctx, A, dt, C=64, sigma=1 if grid else 1024, K=8 if dt == "f16" else 4, offsets=grid, device=True)
    x, b = _vector(_uniform(A.n, seed, 1), dt), _vector(_uniform(A.n, seed, 2), dt)
    y = F.vector(ctx, dt, A.n)
    return {"run": _run_residual if case["op"] == "residual" else _run_operate, "A": A, "S": S, "x": x, "b": b, "y": y,
            "out": _tensor(y, dt)}


def _prepare_cg(case, seed):
    ctx, A = _ctx(), _csr(case, seed)
    S = F.SELL(ctx, A, "f64", C=64, K=4, offsets=True, device=True)
    v = {k: F.vector(ctx, "f64", A.n) for k in ("x", "r", "p", "q")}
    return {"run": _run_cg, "A": A, "S": S, "b": _vector(_uniform(A.n, seed, 1)), "steps": case["steps"], **v,
            "out": _tensor(v["x"], "f64")}


def _prepare_learn(case, seed):
    ctx = _ctx()
    grid = {"matrix": "7v", "nx": case["nx"], "ny": case["nx"], "nz": case["nx"], "peclet": 0.0}
    A = _csr(grid, seed)
    P = F.SDAINV(A, 0.1, 1.0, "f16", ctx=ctx, device=True)
    L = learn.LearnSystem(ctx, A, P, learn.features(A, P, A.diagonal()))
    L.set_probes(torch.stack([_uniform(A.n, seed, 16 + k) for k in range(case["probes"])]).float().cpu().numpy())
    mlp = learn.MLP(ctx, seed=int(seed))
    p = learn.unpack(mlp.get())
    g = torch.Generator().manual_seed(int(seed))   # past the first step the last layer is not zero
    p["w3"] = (0.05 * torch.randn(p["w3"].shape, generator=g)).numpy()
    mlp.set(learn.pack(p))
    return {"run": _run_learn, "keep": (A, P), "L": L, "mlp": mlp, "loss": case["loss"]}


# -------------------------------------------------------------------- run ---
def run(state):
    return state["run"](state)


def _run_solve(s):
    s["x"].fill(0.0)
    r = s["S"].solve(s["b"], s["x"])
    return {"x": s["out"], "solved": int(r.is_solved)}


def _run_batch(s):
    s["x"].fill(0.0)
    r = s["B"].solve(s["bs"], s["xs"])
    return {"x": s["out"], "solved": sum(int(q.is_solved) for q in r)}


def _run_operate(s):
    s["S"].operate(s["x"], s["y"])
    return s["out"]


def _run_residual(s):
    s["S"].compute_residual(s["b"], s["x"], s["y"])
    return s["out"]


def _run_cg(s):
    A, x, r, p, q = s["S"], s["x"], s["r"], s["p"], s["q"]
    x.fill(0.0)
    r.copy(s["b"])
    p.copy(s["b"])
    rr = F.dot(r, r)
    for _ in range(s["steps"]):
        A.operate(p, q)
        alpha = rr / F.dot(p, q)
        x.axpy(alpha, p)
        r.axpy(-alpha, q)
        new = F.dot(r, r)
        p.scale(new / rr).axpy(1.0, r)
        rr = new
    return {"x": s["out"], "rr": rr}


def _run_learn(s):
    s["mlp"].grad_zero()
    loss = s["L"].loss(s["mlp"], grad=True, kind=s["loss"])
    return {"loss": loss, "grad": s["mlp"].grad()}


# ------------------------------------------------------------------- work ---
def _size(case):
    """(rows, entries) of the case's matrix"""
    if case["matrix"] == "graph":
        return case["n"], case["n"] * (case["mean"] + 1)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    if case.get("npts", 7 if case["matrix"] == "7v" else 27) == 7:
        return n, 7 * n - 2 * (nx * ny + ny * nz + nx * nz)
    return n, (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)


def _nest_work(n, nnz, steps, variant="half", values=1.0):
    """the products of `steps` outer steps of the nest m = (100; 8, 4, 2): each
    reads its matrix values once (`values` < 1: shared by several right-hand
    sides) and its vector, and writes one; vector work is left out"""
    inner = {"half": 2, "float": 4, "double": 8}[variant]
    mid = 8 if variant == "double" else 4
    deep = NEST[1] * NEST[2] * steps                # level-3 steps
    by = deep * NEST[3] * (inner * nnz * values + 2 * inner * n)
    by += NEST[1] * steps * (mid * nnz * values + 2 * mid * n) + steps * (8 * nnz * values + 16 * n)
    return {"bytes": by, "flops": 2.0 * nnz * (deep * NEST[3] + NEST[1] * steps + steps)}


def work(case):
    kind = case["kind"]
    if kind == "solve":
        n, nnz = _size(case)
        return _nest_work(n, nnz, STEPS, case["variant"])
    if kind == "nest":
        n, nnz = _size(case)
        deep, mid = 64 * STEPS, 8 * STEPS
        return {"bytes": deep * (2 * nnz + 4 * n) + mid * (4 * nnz + 8 * n) + STEPS * (8 * nnz + 16 * n),
                "flops": 2.0 * nnz * (deep + mid + STEPS)}
    if kind == "batch":
        tot = {"bytes": 0.0, "flops": 0.0}
        for points, edge, margin in _family(case):
            n, nnz = _size(_batch_matrix(points, edge, margin))
            w = _nest_work(n, nnz, 2, values=1.0 / case["rhs"])
            tot = {k: tot[k] + case["rhs"] * w[k] for k in tot}
        return tot
    if kind == "spmv":
        n, nnz = _size(case)
        e = _BYTES[case["dtype"]]
        index = 4 if case["format"] == "csr" or case["matrix"] == "graph" else 0
        return {"bytes": nnz * (e + index) + n * e * (3 if case["op"] == "residual" else 2), "flops": 2.0 * nnz}
    if kind == "cg":
        n, nnz = _size(case)
        return {"bytes": case["steps"] * (8 * nnz + 8 * n * 13), "flops": case["steps"] * (2.0 * nnz + 12.0 * n)}
    n = case["nx"] ** 3
    nnz = 7 * n - 6 * case["nx"] ** 2
    # A, A^T, Z, Z^T and W^T (fp32) once per probe, features and activations once
    return {"bytes": case["probes"] * (2 * 8 * nnz + 3 * 8 * n + 10 * 4 * n) + n * 64,
            "flops": n * (6.0 * (16 * 64 + 64 * 64 + 64)) + case["probes"] * 4.0 * (nnz + n)}


# ------------------------------------------------------------------ exact ---
def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "nest"):
        n, A = _matvec(case, seed)
        x = _solve64(n, A, _uniform(n, seed, 1))
        return None if x is None else {"x": x, "solved": None}
    if kind == "batch":
        parts, at = [], 0
        fam = _family(case)
        rows = [e ** 3 for _, e, _ in fam for _ in range(case["rhs"])]
        b = _uniform(sum(rows), seed, 1)
        for points, edge, margin in fam:
            n, A = _matvec(_batch_matrix(points, edge, margin), seed)
            for _ in range(case["rhs"]):
                x = _solve64(n, A, b[at:at + n])
                if x is None:
                    return None
                parts.append(x)
                at += n
        return {"x": torch.cat(parts), "solved": None}
    if kind == "spmv":
        n, A = _matvec(case, seed)
        dt = _TORCH[case["dtype"]]
        y = A(_uniform(n, seed, 1).to(dt).double())
        return _uniform(n, seed, 2).to(dt).double() - y if case["op"] == "residual" else y
    if kind == "cg":
        n, A = _matvec(case, seed)
        r = _uniform(n, seed, 1)
        x, p, rr = torch.zeros_like(r), r.clone(), torch.dot(r, r)
        for _ in range(case["steps"]):
            q = A(p)
            alpha = rr / torch.dot(p, q)
            x, r = x + alpha * p, r - alpha * q
            new = torch.dot(r, r)
            p, rr = r + (new / rr) * p, new
        return {"x": x, "rr": float(rr)}
    # the SDAINV factors a learned step starts from have no value outside this framework
    return None
