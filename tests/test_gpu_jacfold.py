"""A Jacobi step's x formed by the kernel before it (restriction, defect,
the step before) against a kernel of its own (UGMG_GS_FUSE=0): the same bits,
scalar and in blocks of 2 to 4, both precisions, several columns, one to
three steps, gamma 2 and local levels with inactive vectors."""
import numpy as np
import pytest

from ug_amd import problems, ugmg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cycle(P, monkeypatch, fuse, cols=1, **kw):
    monkeypatch.setenv("UGMG_FUSE_ROWS", "0")
    monkeypatch.setenv("UGMG_GS_FUSE", str(fuse))
    lv = P.levels[-1]
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(P)
    ctx.set_params(**{**dict(nu1=2, nu2=2, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_JAC, damp=0.8,
                             base_abslimit=1e-300, base_maxiter=1), **kw})
    if cols > 1:
        ctx.set_batch(cols)
    ctx.preprocess()
    f = np.random.default_rng(3).uniform(-1.0, 1.0, (cols, lv.n, lv.b))
    for j in range(lv.b):
        f[:, (lv.skip >> j) & 1 == 1, j] = 0.0
    b = torch.from_numpy(f.reshape(cols, -1)).cuda()
    c = torch.zeros_like(b)
    torch.cuda.synchronize()
    for _ in range(2):
        if cols > 1:
            ctx.iter_batch(P.top, c, b)
        else:
            ctx.iter(P.top, c[0], b[0])
    ctx.sync()
    ctx.close()
    return c.cpu().numpy(), b.cpu().numpy()


CASES = [
    (lambda: problems.q1(2, 3, 4, problems.KAPPA_JUMP, seed=1), dict(nu1=1, nu2=1)),
    (lambda: problems.q1(3, 1, 4, problems.KAPPA_JUMP, seed=2), dict(nu1=3, cols=3)),
    (lambda: problems.q1(3, 1, 4, problems.KAPPA_JUMP, seed=3), dict(precision=ugmg.MIXED, nu1=0, gamma=2)),
    (lambda: problems.elasticity(3), dict(precision=ugmg.MIXED)),
    (lambda: problems.elasticity(3), dict(nu2=3, cols=2)),
    (lambda: problems.p1_local(4, 2), {}),
    (lambda: problems.p1_local(3, 2, 2), {}),
    (lambda: problems.p1_local(3, 2, 4), dict(nu1=1, gamma=2)),
    (lambda: problems.elasticity_local(2, 2), dict(precision=ugmg.MIXED)),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_folded_jacobi_steps_are_bitwise_the_separate_ones(k, monkeypatch):
    make, kw = CASES[k]
    P = make()
    print(f"jacfold {k} {[lv.n for lv in P.levels]} b {P.levels[-1].b}", flush=True)
    want, got = (_cycle(P, monkeypatch, f, **kw) for f in (0, 1))
    assert np.all(np.isfinite(want[0])) and np.any(want[0])
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
