"""Large batches of at least four columns on rows of at most 8 entries take
several columns per thread (here, with UGMG_MC_WAVES=0, small ones too, but for
5 columns, whose second group would be mostly empty): cycles and BiCGStab give
every column the bits it gets alone, with full and partial groups of columns,
GS and Jacobi levels, uniform and explicit slices, both precisions."""
import numpy as np
import pytest

from ug_amd import problems, ugmg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _context(P, cols, **kw):
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(P)
    ctx.set_params(**{**dict(nu1=1, nu2=2, gamma=1, baselevel=2, smoother=ugmg.SMOOTH_GS, damp=1.0, base_abslimit=1e-300,
                             base_maxiter=1, inner_cycles=1), **kw})
    ctx.set_batch(cols)
    ctx.preprocess()
    lv = P.levels[-1]
    f = np.random.default_rng(cols).uniform(-1.0, 1.0, (cols, lv.n))
    f[:, lv.skip & 1 == 1] = 0.0
    return ctx, torch.from_numpy(f).cuda()


@pytest.mark.parametrize("cols", [4, 5, 6, 7, 8, 13])
@pytest.mark.parametrize("which,kw", [
    ("cd", {}), ("cd", dict(precision=ugmg.MIXED, damp=0.9)), ("local", dict(baselevel=1)),
    ("q1", dict(smoother=ugmg.SMOOTH_JAC, damp=0.8))])
def test_columns_of_a_cycle(which, kw, cols, monkeypatch):
    monkeypatch.setenv("UGMG_FUSE_ROWS", "0")     # the launches, on small levels too
    monkeypatch.setenv("UGMG_MC_WAVES", "0")
    P = {"cd": lambda: problems.p1_cd(5, 1e-3, float("nan"), seed=1), "local": lambda: problems.p1_local(4, 2),
         "q1": lambda: problems.q1(3, 1, 4, problems.KAPPA_JUMP, seed=2)}[which]()
    print(f"columns {which} {cols}", flush=True)
    ctx, f = _context(P, cols, **kw)
    b, c = f.clone(), torch.zeros_like(f)
    torch.cuda.synchronize()
    ctx.iter_batch(P.top, c, b)
    ctx.sync()
    for j in range(cols):
        if which == "local":      # its coarse defects keep what earlier calls left at VNCLASS < 2
            ctx.close()
            ctx, _ = _context(P, cols, **kw)
        b1, c1 = f[j:j + 1].clone(), torch.zeros_like(f[j:j + 1])
        torch.cuda.synchronize()
        ctx.iter_batch(P.top, c1, b1)
        ctx.sync()
        assert torch.equal(c1[0], c[j]) and torch.equal(b1[0], b[j]), j
    ctx.close()


@pytest.mark.parametrize("cols", [4, 6, 13])
@pytest.mark.parametrize("precision", [ugmg.FP64, ugmg.MIXED])
def test_columns_of_bicgstab(precision, cols, monkeypatch):
    monkeypatch.setenv("UGMG_MC_WAVES", "0")
    P = problems.p1_cd(5, 1e-3, float("nan"), seed=3)
    print(f"bicgstab columns {cols}", flush=True)
    ctx, f = _context(P, cols, precision=precision, nu2=1)
    f[1] *= 1e-3
    f[2] = 0.0                                     # done at once
    b, x = f.clone(), torch.zeros_like(f)
    torch.cuda.synchronize()
    res, _ = ctx.bcgs(P.top, x, b, red=1e-8, maxiter=60)
    ctx.sync()
    for j in range(cols):
        b1, x1 = f[j:j + 1].clone(), torch.zeros_like(f[j:j + 1])
        torch.cuda.synchronize()
        r1, _ = ctx.bcgs(P.top, x1, b1, red=1e-8, maxiter=60)
        ctx.sync()
        assert r1[0].number_of_linear_iterations == res[j].number_of_linear_iterations
        assert torch.equal(x1[0], x[j]), j
    ctx.close()
