"""What is measured of the multigrid solve path: the calls a program that links
it makes, over the sizes it makes them at.

A case is a dict of plain values; `kind` names the entry point:

  smooth  one smoothing step on a level (ugmg_jacobi_step / ugmg_gs_step)
  cycle   one lmgc cycle as a preconditioner (ugmg_iter, ugmg_iter_batch)
  ls      a whole linear solve, ls + lmgc (ugmg_solve)
  surface the solve on a locally refined hierarchy (ugmg_solve_surface)
  bcgs    BiCGStab over the cycle, several right-hand sides (ugmg_bcgs_solve)
  setup   a new matrix: levels in, preprocess, the first cycle
  serve   a burst of requests to the solve server

`problem` and its sizes: q1 (Q1 Poisson or jump coefficient on `cells`
coarse cells per direction refined `nref` times, `dim` 2 or 3), cd2d (SUPG P1
convection-diffusion), elast (P1 elasticity, 3x3 blocks), local (the same,
refined toward a corner).  Sizes, parameters and stop limits are those of the
benchmark's legs and of the GPU tests, with odd cell counts besides.
"""
from __future__ import annotations

import functools

import numpy as np
import torch

from ug_amd import problems, ugmg

LOAD_SEED = 0x5EED0004     # the locally refined case's load stream starts here


# ------------------------------------------------------------------- cases
def listed():
    return [
        # smallest call: a V(1,1) Jacobi cycle on 65^2, the preconditioner of
        # a small 2D Krylov solve; launches and latency
        dict(name="cycle_2d_65", kind="cycle", problem="q1", dim=2, cells=2, nref=5, jump=False, smoother="jac",
             nu=1, base=1, prec="fp64", cols=1),
        # a few load cases of one 33^3 jump-coefficient matrix at once
        dict(name="cycle_3d_33_cols8", kind="cycle", problem="q1", dim=3, cells=1, nref=5, jump=True, smoother="gs",
             nu=2, base=3, prec="fp64", cols=8),
        # damped Jacobi on a large 2D grid: a bandwidth-bound layer
        dict(name="jac_2d_1025", kind="smooth", problem="q1", dim=2, cells=2, nref=9, jump=True, smoother="jac"),
        # multicolour Gauss-Seidel on the finest level of the headline problem
        dict(name="gs_3d_129", kind="smooth", problem="q1", dim=3, cells=1, nref=7, jump=True, smoother="gs"),
        # the benchmark's 2D Poisson solve
        dict(name="ls_poisson_2d_129", kind="ls", problem="q1", dim=2, cells=2, nref=6, jump=False, smoother="jac",
             nu=2, base=0, prec="fp64", red=1e-10),
        # a mid-sized FP64 solve
        dict(name="ls_jump_3d_65", kind="ls", problem="q1", dim=3, cells=1, nref=6, jump=True, smoother="gs",
             nu=2, base=4, prec="fp64", red=1e-10),
        # the headline solve
        dict(name="ls_jump_3d_129_mixed", kind="ls", problem="q1", dim=3, cells=1, nref=7, jump=True,
             smoother="gs", nu=2, base=4, prec="mixed", red=1e-10),
        # 3x3 blocks: the uniform elasticity leg
        dict(name="ls_elast_65_mixed", kind="ls", problem="elast", nref=6, smoother="gs", nu=2, base=3,
             prec="mixed", red=1e-10),
        # the locally refined elasticity leg
        dict(name="surface_elast_33_3", kind="surface", problem="local", nref=5, depth=3, smoother="jac", nu=2,
             base=3, prec="mixed", red=1e-8),
        # 32 right-hand sides of a nonsymmetric problem
        dict(name="bcgs_cd2d_513_32", kind="bcgs", problem="cd2d", nref=8, smoother="gs", nu=1, base=3,
             prec="mixed", cols=32, red=1e-8),
        # a new matrix every nonlinear step
        dict(name="setup_jump_3d_65", kind="setup", problem="q1", dim=3, cells=1, nref=6, jump=True, smoother="gs",
             nu=2, base=4, prec="fp64", cols=1, source="levels"),
        # twelve requests of four shapes at once, groups resident
        dict(name="serve_12", kind="serve", problem="q1", requests=12, nref2=6, nref3=5, red=1e-8),
    ]


def draw(rng):
    kind = rng.choice(["smooth", "smooth", "cycle", "cycle", "cycle", "ls", "ls", "ls", "surface", "bcgs", "bcgs",
                       "setup", "serve"])
    if kind == "serve":
        return dict(kind=kind, problem="q1", requests=rng.randint(2, 12), nref2=rng.randint(4, 6),
                    nref3=rng.randint(3, 5), red=10.0 ** -rng.randint(6, 9))
    if kind == "surface":
        nref, depth = rng.choice([(2, 2), (3, 1), (3, 2), (3, 3), (4, 1), (4, 2)])
        return dict(kind=kind, problem="local", nref=nref, depth=depth, smoother="jac", nu=rng.randint(1, 3),
                    base=rng.randint(1, 2), prec=rng.choice(["fp64", "mixed"]), red=10.0 ** -rng.randint(6, 9))
    if kind == "bcgs":
        nref = rng.randint(4, 8)
        return dict(kind=kind, problem="cd2d", nref=nref, smoother="gs", nu=rng.randint(1, 2),
                    base=rng.randint(1, 3), prec=rng.choice(["fp64", "mixed"]), cols=rng.randint(1, 32 if nref < 8 else 20),
                    red=10.0 ** -rng.randint(6, 9))
    if kind == "ls" and rng.random() < 0.3:
        nref = rng.randint(3, 5)
        return dict(kind=kind, problem="elast", nref=nref, smoother=rng.choice(["gs", "jac"]), nu=rng.randint(1, 3),
                    base=rng.randint(1, nref - 2), prec=rng.choice(["fp64", "mixed"]), red=10.0 ** -rng.randint(8, 10))
    # Q1 grids: any cell count, the level sizes spread over their logarithm
    dim = rng.choice([2, 2, 3, 3, 3])
    # whole 2D solves with a jumping coefficient are no work for this cycle
    # (hundreds of iterations or none that converge)
    jump = kind == "smooth" or rng.random() < (0.0 if kind == "ls" and dim == 2 else 0.75)
    most = {2: 1025, 3: 129 if kind == "smooth" else 97}[dim] if kind != "setup" else {2: 513, 3: 65}[dim]
    sizes = [(c, r) for c in (1, 2, 3, 5, 7) for r in range(2, 11) if (9 if dim == 3 else 17) <= c * 2 ** r + 1 <= most]
    want = (9 if dim == 3 else 17) * (most / (9 if dim == 3 else 17)) ** rng.random()
    cells, nref = min(sizes, key=lambda s: abs(np.log((s[0] * 2 ** s[1] + 1) / want)) + 0.2 * rng.random())
    case = dict(kind=kind, problem="q1", dim=dim, cells=cells, nref=nref, jump=jump,
                smoother="gs" if dim == 3 or rng.random() < 0.5 else "jac")
    if kind == "smooth":
        return case
    # the base level: at most 17^3 or 33^2 vectors, at least one below the top
    fits = [l for l in range(nref) if (cells * 2 ** l + 1) ** dim <= (4913 if dim == 3 else 1100)]
    case.update(nu=rng.randint(1, 3), base=rng.choice(fits[-2:]),
                prec="fp64" if kind == "setup" or rng.random() < 0.5 else "mixed")
    if kind == "ls":
        return dict(case, nu=2, red=10.0 ** -rng.randint(8, 10))
    cols = rng.choice([1, 1, 2, 3, 5, 8]) if kind == "cycle" and case["prec"] == "fp64" and nref < 7 else 1
    if kind == "setup":
        return dict(case, cols=1, source=rng.choice(["levels", "elements"]))
    return dict(case, cols=cols)


# ---------------------------------------------------------------- problems
@functools.lru_cache(maxsize=2)
def _fixed(problem, nref, depth):
    """The elasticity hierarchies: their matrices do not depend on a seed."""
    return problems.elasticity(nref) if problem == "elast" else problems.elasticity_local(nref, depth)


def _problem(case, seed):
    if case["problem"] == "q1":
        kappa = problems.KAPPA_JUMP if case["jump"] else problems.KAPPA_ONE
        return problems.q1(case["dim"], case["cells"], case["nref"], kappa, seed=seed + 1)
    if case["problem"] == "cd2d":
        return problems.p1_cd(case["nref"], 1e-3, float("nan"), seed=seed + 1)
    return _fixed(case["problem"], case["nref"], case.get("depth", 0))


def _params(case):
    gs = case["smoother"] == "gs"
    return dict(nu1=case.get("nu", 2), nu2=case.get("nu", 2), gamma=1, baselevel=case["base"] if "base" in case else _top_base(case),
                smoother=ugmg.SMOOTH_GS if gs else ugmg.SMOOTH_JAC, damp=1.0 if gs else 0.8, base_abslimit=1e-300,
                base_red=1e-12, base_maxiter=1, use_graph=1,
                precision=ugmg.MIXED if case.get("prec") == "mixed" else ugmg.FP64,
                inner_cycles=1 if case["kind"] in ("bcgs", "cycle") else 7)


def _top_base(case):
    """The base level of a hierarchy set up for single smoothing steps."""
    return max(l for l in range(case["nref"]) if (case["cells"] * 2 ** l + 1) ** case["dim"] <= 1100)


def _loads(lv, cols, seed):
    """Right-hand sides ~U[-1, 1], 0 on Dirichlet components: (cols, n*b)."""
    f = np.random.default_rng(seed).uniform(-1.0, 1.0, (cols, lv.n, lv.b))
    for j in range(lv.b):
        f[:, (lv.skip >> j) & 1 == 1, j] = 0.0
    return torch.from_numpy(f.reshape(cols, -1))


def _context(case, P, stream):
    ctx = ugmg.Context(0)
    ctx.set_stream(stream)
    ctx.set_hierarchy(P)
    ctx.set_params(**_params(case))
    if case.get("cols", 1) > 1:
        ctx.set_batch(case["cols"])
    return ctx


# --------------------------------------------------------------- preparing
def _request_problems(case, seed):
    """The requests of a burst: 2D Poisson and 3D jump-coefficient problems,
    each shape at its finest size and one below."""
    out = []
    for i in range(case["requests"]):
        if i % 2 == 0:
            out.append(problems.q1(2, 2, case["nref2"] - i // 2 % 2, problems.KAPPA_ONE, seed=100 * seed + i + 1))
        else:
            out.append(problems.q1(3, 1, case["nref3"] - i // 2 % 2, problems.KAPPA_JUMP, seed=100 * seed + i + 1))
    return out


def _prepare_serve(case, seed):
    reqs = []
    for P in _request_problems(case, seed):
        bl = max(l for l in range(P.top + 1) if P.levels[l].n <= 300)
        reqs.append((P, ugmg.default_params(nu1=2, nu2=2, gamma=1, baselevel=bl, smoother=ugmg.SMOOTH_GS, damp=1.0,
                                            base_abslimit=1e-300, use_graph=1)))
    srv = ugmg.Server(0, budget_bytes=64e9, max_slots=8)
    state = dict(case=case, srv=srv, reqs=reqs, done=0)
    run(state)      # a server that has been up for a while: its groups are resident
    return state


def prepare(case, seed):
    if case["kind"] == "serve":
        return _prepare_serve(case, seed)
    P = _problem(case, seed)
    lv = P.levels[-1]
    stream = torch.cuda.Stream()
    ctx = _context(case, P, stream)
    state = dict(case=case, P=P, ctx=ctx, stream=stream, top=P.top)
    if case["kind"] == "setup":
        state["rhs"] = _loads(lv, 1, seed).cuda()
        if case["source"] == "elements":
            el = problems.q1_elements(case["dim"], case["cells"], case["nref"],
                                      problems.KAPPA_JUMP if case["jump"] else problems.KAPPA_ONE, seed=seed + 1)
            state["el"] = dict(n=el.n, elem=torch.from_numpy(el.elem).cuda(), kref=torch.from_numpy(el.kref).cuda(),
                               scale=torch.from_numpy(el.scale).cuda(),
                               skip=torch.from_numpy(el.skip.view(np.int32)).cuda())
        state["x"], state["b"] = torch.zeros_like(state["rhs"]), torch.empty_like(state["rhs"])
        torch.cuda.synchronize()
        return state
    ctx.preprocess()
    if case["kind"] == "surface":
        load = problems.surface_load(P, case["base"], LOAD_SEED + 1000 * seed)
        state["rhs"] = [None if f is None else torch.from_numpy(f).cuda() for f in load]
        state["x"] = [None if f is None else torch.zeros_like(f) for f in state["rhs"]]
        state["b"] = [None if f is None else torch.empty_like(f) for f in state["rhs"]]
    else:
        state["rhs"] = _loads(lv, case.get("cols", 1), seed).cuda()
        state["x"], state["b"] = torch.zeros_like(state["rhs"]), state["rhs"].clone()
    torch.cuda.synchronize()
    return state


# ------------------------------------------------------------------- a pass
def _run_serve(s):
    srv, c = s["srv"], s["case"]
    ids = [srv.submit(P, prm, red=c["red"], maxiter=500) for P, prm in s["reqs"]]
    s["done"] += len(ids)
    srv.drain(s["done"])
    return [srv.result(i, P.levels[-1].n) for i, (P, _) in zip(ids, s["reqs"])]


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "serve":
        return _run_serve(s)
    ctx, top = s["ctx"], s["top"]
    if kind == "smooth":    # steps follow one another on one defect
        (ctx.gs_step if c["smoother"] == "gs" else ctx.jacobi_step)(top, s["x"][0], s["b"][0])
        return {"x": s["x"], "b": s["b"]}
    with torch.cuda.stream(s["stream"]):
        if kind == "surface":
            for x, b, f in zip(s["x"], s["b"], s["rhs"]):
                if f is not None:
                    x.zero_()
                    b.copy_(f)
            ctx.solve_surface(top, s["x"], s["b"], red=c["red"], maxiter=200, record=False)
            return {"x": [x for x in s["x"] if x is not None]}
        s["b"].copy_(s["rhs"])
        if kind == "cycle":     # c := correction, b -= A c
            if c["cols"] > 1:
                ctx.iter_batch(top, s["x"], s["b"])
            else:
                ctx.iter(top, s["x"][0], s["b"][0])
            return {"c": s["x"], "b": s["b"]}
        if kind == "setup":
            if c["source"] == "elements":
                el = s["el"]
                ctx.assemble_level(top, el["n"], el["elem"], kref=el["kref"], scale=el["scale"], skip=el["skip"])
                for l in range(top, c["base"], -1):
                    ctx.galerkin(l)
            else:
                ctx.set_hierarchy(s["P"])
            ctx.preprocess()
            ctx.iter(top, s["x"][0], s["b"][0])
            return {"c": s["x"], "b": s["b"]}
        s["x"].zero_()
        if kind == "bcgs":
            ctx.bcgs(top, s["x"], s["b"], red=c["red"], maxiter=200, maxdef=1)
        else:
            ctx.solve(top, s["x"][0], s["b"][0], red=c["red"], maxiter=500, record=False)
        # the final defect is the rounding of the last iterations: its digits
        # lie below the stop limit, so the solution alone is the answer
        return {"x": s["x"]}


# --------------------------------------------------------------------- work
def _sizes(case):
    """(unknown vectors, matrix blocks) of every level, coarsest first."""
    out = []
    for l in range(case["nref"] + 1):
        if case["problem"] == "q1":
            m, d = case["cells"] * 2 ** l + 1, case["dim"]
            out.append((m ** d, (3 * m - 2) ** d))
        elif case["problem"] == "cd2d":
            m = 2 ** (l + 1) + 1
            out.append((m * m, 7 * m * m))
        else:
            m = 2 ** l + 1
            out.append((m ** 3, 15 * m ** 3))
    return out + [out[-1]] * case.get("depth", 0)    # local levels: about the finest uniform one's size


def work(case):
    """Per smoothing step one pass over a level's matrix (values; a stencil
    needs no index per entry) and over x, b and c; a cycle has nu + nu steps
    and the defect of the coarse correction on every level above the base."""
    if case["kind"] == "serve":
        by = fl = 0.0
        for i in range(case["requests"]):
            dim = 2 + i % 2
            sub = dict(kind="ls", problem="q1", dim=dim, cells=4 - dim, jump=dim == 3, base=2, nu=2, prec="fp64",
                       nref=(case["nref2"] if dim == 2 else case["nref3"]) - i // 2 % 2)
            w = work(sub)
            by, fl = by + w["bytes"], fl + w["flops"]
        return {"bytes": by, "flops": fl}
    bb = 9 if case["problem"] in ("elast", "local") else 1
    nb = 3 if bb == 9 else 1
    sz = _sizes(case)
    v = 4 if case.get("prec") == "mixed" else 8
    cols = case.get("cols", 1)
    if case["kind"] == "smooth":
        n, nnz = sz[-1]
        return {"bytes": 8.0 * (nnz + 4 * n), "flops": 2.0 * nnz}
    passes = 2 * case["nu"] + 1
    by = sum(passes * v * (nnz * bb + 4.0 * n * nb * cols) for n, nnz in sz[case["base"] + 1:])
    by += v * (sz[case["base"]][0] * nb) ** 2
    fl = sum(passes * 2.0 * nnz * bb * cols for n, nnz in sz[case["base"] + 1:])
    if case["kind"] == "setup":     # the levels come in, their layouts go out
        by += sum(2 * 12.0 * nnz * bb for n, nnz in sz[case["base"]:])
        return {"bytes": by, "flops": fl}
    # cycles to the stop limit: per decade of reduction, about 1 for Poisson
    # and convection-diffusion, 4 to 5 for jumps and elasticity
    if case["kind"] in ("ls", "surface", "bcgs"):
        decades = -np.log10(case.get("red", 1e-8))
        per = 1.0 if case["kind"] == "bcgs" or case["problem"] == "q1" and not case["jump"] else 4.5
        its = np.ceil(decades * per) * (2 if case["kind"] == "bcgs" else 1)
        by, fl = by * its, fl * its
    return {"bytes": float(by), "flops": float(fl)}


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times what the path is off by from the same in 64 bits
    with sums in another order; solves that a rounding can move within their
    stop limit (FP32 cycles, BiCGStab), from another route to that limit."""
    if case["kind"] in ("smooth", "cycle", "setup"):
        if case.get("prec") == "mixed":
            return {"rel": 4e-6, "max": 4e-4}
        return {"rel": 1e-13, "max": 1e-10}
    if case.get("prec") == "mixed" or case["kind"] == "bcgs":
        return {"rel": 12 * case["red"], "max": 1000 * case["red"]}
    return {"rel": 1e-10, "max": 1e-7}


# -------------------------------------------------------- the same in 64 bits
def _matrix(lv):
    """Scalar CSR (torch, float64) of a level."""
    b = lv.b
    rp, ci, va = lv.row_ptr.astype(np.int64), lv.col_idx.astype(np.int64), lv.vals
    if b > 1:
        rows = np.repeat(np.arange(lv.n), np.diff(rp))
        r = (rows[:, None, None] * b + np.arange(b)[None, :, None]) + np.zeros((1, 1, b), np.int64)
        c = ci[:, None, None] * b + np.arange(b)[None, None, :] + np.zeros((1, b, 1), np.int64)
        m = torch.sparse_coo_tensor(np.stack([r.ravel(), c.ravel()]), torch.from_numpy(va), (lv.n * b, lv.n * b))
        return m.coalesce().to_sparse_csr()
    return torch.sparse_csr_tensor(torch.from_numpy(rp), torch.from_numpy(ci), torch.from_numpy(va), (lv.n, lv.n))


def _prolongation(lv, nc):
    return torch.sparse_csr_tensor(torch.from_numpy(lv.p_ptr.astype(np.int64)),
                                   torch.from_numpy(lv.p_idx.astype(np.int64)), torch.from_numpy(lv.p_w), (lv.n, nc))


def _colours(lv, dim):
    """First-fit colours of a 9- or 27-point grid: the parities."""
    m, i = lv.nodes_per_dir, torch.arange(lv.n)
    col = i % m % 2 + 2 * (i // m % m % 2)
    return col if dim == 2 else col + 4 * (i // (m * m) % 2)


def _step(A, diag, col, b, damp):
    """x and the new defect of one smoothing step; b: (n, columns)."""
    if col is None:
        x = damp * b / diag
        return x, b - A @ x
    x = torch.zeros_like(b)
    for k in range(int(col.max()) + 1):
        at = col == k
        x[at] = ((b - A @ x) / diag)[at]
    return x, b - A @ x


def _cycle(case, mats, levels, l, b):
    if l == case["base"]:
        c = torch.linalg.solve(mats[l].to_dense(), b)
        return c, b - mats[l] @ c
    A, lv, low = mats[l], levels[l], levels[l - 1]
    diag = torch.from_numpy(lv.vals[lv.row_ptr[:-1]]) if mats[l] is not None else None
    if case.get("source") == "elements":
        diag = _diagonal(A)
    diag = diag[:, None]
    gs = case["smoother"] == "gs"
    col = _colours(lv, case["dim"]) if gs else None
    damp = 1.0 if gs else 0.8
    c = torch.zeros_like(b)
    for _ in range(case["nu"]):
        x, b = _step(A, diag, col, b, damp)
        c = c + x
    P = _prolongation(lv, low.n)
    bc = P.t() @ b
    bc[torch.from_numpy(low.skip == 1)] = 0.0
    cc, _ = _cycle(case, mats, levels, l - 1, bc)
    t = P @ cc
    t[torch.from_numpy(lv.skip == 1)] = 0.0
    c, b = c + t, b - A @ t
    for _ in range(case["nu"]):
        x, b = _step(A, diag, col, b, damp)
        c = c + x
    return c, b


def _diagonal(A):
    rows = torch.repeat_interleave(torch.arange(A.shape[0]), A.crow_indices().diff())
    at = rows == A.col_indices()
    d = torch.zeros(A.shape[0], dtype=torch.float64)
    d[rows[at]] = A.values()[at]
    return d


def _cg(A, f, most=4000):
    """Conjugate gradients with the diagonal, to the rounding of 64 bits; the
    loads vanish on the Dirichlet rows, where the iterates stay 0."""
    d = _diagonal(A)
    x, r = torch.zeros_like(f), f.clone()
    z = r / d
    p, rz, stop = z.clone(), float(r @ z), 1e-14 * float(torch.linalg.norm(f))
    for _ in range(most):
        q = A @ p
        a = rz / float(p @ q)
        x += a * p
        r -= a * q
        if float(torch.linalg.norm(r)) < stop:
            break
        z = r / d
        rz, old = float(r @ z), rz
        p = z + (rz / old) * p
    return x


def _grid_solve(A, m, f):
    """Direct solution on an m x m grid (rows of the grid coupled to the next
    ones only): block elimination over the grid rows; f: (columns, m*m)."""
    rows = torch.repeat_interleave(torch.arange(A.shape[0]), A.crow_indices().diff())
    cols, va = A.col_indices(), A.values()

    def block(i, j):
        at = slice(int(A.crow_indices()[i * m]), int(A.crow_indices()[(i + 1) * m]))
        r, c, v = rows[at] - i * m, cols[at] - j * m, va[at]
        ok = (c >= 0) & (c < m)
        out = torch.zeros(m, m, dtype=torch.float64)
        out[r[ok], c[ok]] = v[ok]
        return out

    g = f.t().reshape(m, m, -1).clone()
    up = []
    for i in range(m):
        D = block(i, i)
        if i > 0:
            low = block(i, i - 1)
            D -= low @ up[-1]
            g[i] -= low @ g[i - 1]
        lu = torch.linalg.lu_factor(D)
        g[i] = torch.linalg.lu_solve(*lu, g[i])
        up.append(torch.linalg.lu_solve(*lu, block(i, i + 1)) if i + 1 < m else None)
    for i in range(m - 2, -1, -1):
        g[i] -= up[i] @ g[i + 1]
    return g.reshape(m * m, -1).t().contiguous()


def _solution(P, f):
    """A x = f on the finest level; None where it would take too long."""
    lv = P.levels[-1]
    A = _matrix(lv)
    if P.dim == 2 and lv.b == 1:
        return _grid_solve(A, lv.nodes_per_dir, f)
    if lv.n * lv.b > 300000:
        return None
    return torch.stack([_cg(A, f[j]) for j in range(f.shape[0])])


def exact(case, seed):
    kind = case["kind"]
    if kind == "surface":
        # the composite solution is defined by the multilevel iteration
        # itself: no direct form without its level-by-level defects
        return None
    if kind == "serve":
        return [_solution(P, torch.from_numpy(P.rhs)[None])[0] for P in _request_problems(case, seed)]
    P = _problem(case, seed)
    lv = P.levels[-1]
    f = _loads(lv, case.get("cols", 1), seed)
    if kind in ("ls", "bcgs"):
        x = _solution(P, f)
        return None if x is None else {"x": x}
    if kind == "smooth":
        diag = torch.from_numpy(lv.vals[lv.row_ptr[:-1]])[:, None]
        gs = case["smoother"] == "gs"
        x, b = _step(_matrix(lv), diag, _colours(lv, case["dim"]) if gs else None, f.t().contiguous(),
                     1.0 if gs else 0.8)
        return {"x": x.t().contiguous(), "b": b.t().contiguous()}
    mats = [None] * case["base"] + [_matrix(l) for l in P.levels[case["base"]:]]
    if case.get("source") == "elements":     # the coarse matrices are P^T A P
        for l in range(P.top, case["base"], -1):
            T = _prolongation(P.levels[l], P.levels[l - 1].n)
            mats[l - 1] = torch.sparse.mm(torch.sparse.mm(T.t().to_sparse_csr(), mats[l]), T)
    c, b = _cycle(case, mats, P.levels, P.top, f.t().contiguous())
    return {"c": c.t().contiguous(), "b": b.t().contiguous()}
