"""ugmg_iter and ugmg_iter_batch replay their cycle from a graph from the
second call on (use_graph): every call, with other vectors and changing
levels, columns and parameters in between, gives the bits of launches."""
import numpy as np
import pytest

from ug_amd import problems, ugmg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kw", [
    dict(smoother=ugmg.SMOOTH_JAC, damp=0.8), dict(), dict(precision=ugmg.MIXED, inner_cycles=2),
    dict(smoother=ugmg.SMOOTH_JAC, damp=0.7, precision=ugmg.MIXED, inner_cycles=1)])
def test_iter_calls(kw):
    P = problems.q1(2, 3, 4, problems.KAPPA_JUMP, seed=1)
    ctxs = []
    for use in (0, 1):
        ctx = ugmg.Context(0)
        ctx.set_stream(torch.cuda.Stream())
        ctx.set_hierarchy(P)
        ctx.set_batch(3)
        ctxs.append(ctx)

    def params(nu):
        for use, ctx in enumerate(ctxs):
            ctx.set_params(**{**dict(nu1=nu, nu2=nu, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_GS, damp=1.0,
                                     base_abslimit=1e-300, base_maxiter=1, use_graph=use), **kw})
            if nu == 1:
                ctx.preprocess()

    params(1)
    # (level, columns) of the calls; then the same with other parameters
    for nu in (1, 2):
        if nu == 2:
            params(2)
        for k, (level, cols) in enumerate([(4, 1), (4, 1), (4, 1), (4, 3), (4, 3), (3, 1), (3, 1), (4, 1), (4, 1)]):
            lv = P.levels[level]
            f = np.random.default_rng(100 * nu + k).uniform(-1.0, 1.0, (cols, lv.n))
            f[:, lv.skip & 1 == 1] = 0.0
            out = []
            for ctx in ctxs:
                b = torch.from_numpy(f).cuda()
                c = torch.zeros_like(b)
                torch.cuda.synchronize()
                if cols > 1:
                    ctx.iter_batch(level, c, b)
                else:
                    ctx.iter(level, c[0], b[0])
                ctx.sync()
                out.append((c.cpu().numpy(), b.cpu().numpy()))
            assert np.any(out[0][0])
            assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]), (nu, k)
    for ctx in ctxs:
        ctx.close()
