"""Device-side EXPreProcess (np/procs/iter.cc:8685-8970): the band LU without
pivoting (EXDecomposeMatrixDOUBLE, gm/evm.cc:1400-1418) and the explicit
inverse from EXApplyLUDOUBLE (gm/evm.cc:1493-1510) run on the GPU during
ugmg_preprocess (for base levels above about 5e7 multiply-adds of
factorisation; UGMG_BASE_HOST=0 forces it for the small levels here).  The
inverse is read back column by column through the
base solve (ls over ex, one step, damp 1, on unit vectors: the GEMV returns
the column exactly) and must be bit-identical to the host factorisation
(UGMG_BASE_HOST=1, and for scalar levels ugmg_coarse_inverse, which the
CPU tests pin against the oracle's EX).  A zero pivot fails on the device
as on the host."""
import os

import numpy as np
import pytest

from ug_amd import problems, ugmg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _context(P, bl, host_factor, reorder=1, ex_float=0):
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(P)
    ctx.set_params(nu1=1, nu2=1, baselevel=bl, smoother=ugmg.SMOOTH_JAC, damp=0.8, base_abslimit=1e-300,
                   base_maxiter=1, ex_reorder=reorder, ex_float=ex_float)
    # small base levels are factored on the host unless forced to the device
    os.environ["UGMG_BASE_HOST"] = "1" if host_factor else "0"
    try:
        ctx.preprocess()
    finally:
        os.environ.pop("UGMG_BASE_HOST", None)
    return ctx


def _inverse_columns(ctx, n):
    inv = np.empty((n, n))
    c = torch.zeros(n, dtype=torch.float64, device="cuda")
    b = torch.zeros(n, dtype=torch.float64, device="cuda")
    for u in range(n):
        b.zero_()
        b[u] = 1.0
        torch.cuda.synchronize()      # the context works on its own stream
        ctx.base_solve(c, b)
        ctx.sync()
        inv[:, u] = c.cpu().numpy()
    return inv


@pytest.mark.parametrize("which", ["jump3d", "poisson2d", "elasticity"])
def test_device_base_inverse_is_bitwise_the_host_one(which):
    if which == "jump3d":
        P, bl = problems.jump3d(4, seed=11), 3          # 9^3 vectors, BFS bandwidth 259
    elif which == "poisson2d":
        P, bl = problems.q1(2, 2, 5, problems.KAPPA_ONE, seed=12), 4   # 33^2 vectors
    else:
        P, bl = problems.elasticity(3, seed=13), 2       # 5^3 vectors x 3 components
    lv = P.levels[bl]
    n = lv.n * lv.b
    dev = _context(P, bl, host_factor=False)
    host = _context(P, bl, host_factor=True)
    got = _inverse_columns(dev, n)
    want = _inverse_columns(host, n)
    dev.close()
    host.close()
    assert np.array_equal(got, want)
    if lv.b == 1:
        rc, inv, _, _ = ugmg.coarse_inverse(lv, reorder=1)
        assert rc == 0 and np.array_equal(got, inv)
    # and it is the inverse
    A = lv.dense()
    assert np.max(np.abs(got @ A - np.eye(n))) < 1e-10


@pytest.mark.parametrize("n,bw", [(1, 0), (40, 1), (97, 16), (64, 31), (65, 32), (100, 33), (353, 48), (450, 420),
                                  (700, 640), (1000, 960), (1100, 1000)])
@pytest.mark.parametrize("ex_float", [0, 1])
def test_device_base_band_widths(n, bw, ex_float):
    """Every path of the factorisation and of the substitutions (panels from a
    half bandwidth of 32 to 992, the LDS window with 32, 20 and 16 columns, the
    general kernels outside) at the edges of its panels and chunks."""
    rng = np.random.default_rng(n)
    offs = sorted({o for d in {1, bw // 2, bw} for o in (-d, d) if d})
    cols = [[v] + [v + o for o in offs if 0 <= v + o < n] for v in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    vals = rng.uniform(-1.0, 1.0, rp[-1])
    vals[rp[:-1]] += 8.0
    lv = problems.Level(n=n, b=1, row_ptr=rp, col_idx=np.concatenate(cols).astype(np.int32), vals=vals,
                        skip=np.zeros(n, np.uint32), vclass=np.full(n, 3, np.uint8), vnclass=np.zeros(n, np.uint8))
    P = problems.Problem(dim=1, levels=[lv])
    dev, host = (_context(P, 0, h, reorder=0, ex_float=ex_float) for h in (False, True))
    c, b = (torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(2))
    for u in sorted({0, n // 3, n - 17, n - 1} & set(range(n))):
        got = []
        for ctx in (dev, host):
            b.zero_()
            b[u] = 1.0
            torch.cuda.synchronize()
            ctx.base_solve(c, b)
            ctx.sync()
            got.append(c.cpu().numpy())
        assert np.array_equal(*got)
    dev.close()
    host.close()


@pytest.mark.parametrize("host_factor", [False, True])
def test_device_base_zero_pivot_fails_like_the_host(host_factor):
    P = problems.q1(2, 2, 1, problems.KAPPA_ONE, seed=1)
    lv = P.levels[0]
    lv.vals = lv.vals.copy()
    lv.vals[lv.row_ptr[0]] = 0.0      # first pivot of the list order
    ctx = _context(P, 0, host_factor=host_factor, reorder=0)
    c = torch.zeros(lv.n, dtype=torch.float64, device="cuda")
    b = torch.ones(lv.n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with pytest.raises(ugmg.UgmgError) as e:
        ctx.base_solve(c, b)
    assert e.value.code == -5
    ctx.close()


def _float_band_lu_inverse(A, bw):
    """EXDecomposeMatrixFLOAT restated in numpy float32 (no pivoting, band
    only), then the inverse from the FLOAT factors in float64 (what
    EXApplyLUFLOAT computes on unit vectors, up to summation order)."""
    import scipy.linalg as sl
    M = A.astype(np.float32)
    n = len(M)
    for i in range(n - 1):
        e = min(i + bw, n - 1) + 1
        f = M[i + 1:e, i] / M[i, i]
        M[i + 1:e, i] = f
        M[i + 1:e, i + 1:e] = M[i + 1:e, i + 1:e] - np.outer(f, M[i, i + 1:e])
    F = M.astype(np.float64)
    L = np.tril(F, -1) + np.eye(n)
    U = np.triu(F)
    return sl.solve_triangular(U, sl.solve_triangular(L, np.eye(n), lower=True, unit_diagonal=True))


def test_ex_float_mode():
    """ex $f (EXInit's $f, np/procs/iter.cc:8253; factors by
    EXDecomposeMatrixFLOAT, applied by EXApplyLUFLOAT)."""
    P, bl = problems.jump3d(4, seed=14), 3
    lv = P.levels[bl]
    n = lv.n
    dev = _context(P, bl, host_factor=False, ex_float=1)
    host = _context(P, bl, host_factor=True, ex_float=1)
    dbl = _context(P, bl, host_factor=False, ex_float=0)
    got, want_host, inv64 = _inverse_columns(dev, n), _inverse_columns(host, n), _inverse_columns(dbl, n)
    for c in (dev, host, dbl):
        c.close()
    assert np.array_equal(got, want_host)
    rc, _, order, bw = ugmg.coarse_inverse(lv, reorder=1)
    assert rc == 0
    A = lv.dense()[np.ix_(order, order)]
    ref = np.empty_like(got)
    ref[np.ix_(order, order)] = _float_band_lu_inverse(A, bw)
    scale = np.max(np.abs(ref))
    assert np.max(np.abs(got - ref)) < 1e-10 * scale
    # FLOAT factors: the inverse differs from the DOUBLE one at float level
    assert 1e-9 < np.max(np.abs(got - inv64)) / scale < 1e-3
