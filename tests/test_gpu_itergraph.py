"""ugmg_iter and ugmg_iter_batch replay their cycle from a graph from the
second call on (use_graph), where it is enough launches: every call, with other
vectors and changing levels, columns and parameters in between, gives the bits
of launches."""
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
        for k, (level, cols) in enumerate([(4, 1), (4, 1), (4, 1), (4, 3), (4, 3), (3, 1), (3, 1), (4, 1), (4, 1),
                                           (4, 0), (4, 1), (4, 0), (4, 0)]):     # 0: a batch of one
            lv = P.levels[level]
            f = np.random.default_rng(100 * nu + k).uniform(-1.0, 1.0, (max(cols, 1), lv.n))
            f[:, lv.skip & 1 == 1] = 0.0
            out = []
            for ctx in ctxs:
                b = torch.from_numpy(f).cuda()
                c = torch.zeros_like(b)
                torch.cuda.synchronize()
                if cols != 1:
                    ctx.iter_batch(level, c, b)
                else:
                    ctx.iter(level, c[0], b[0])
                ctx.sync()
                out.append((c.cpu().numpy(), b.cpu().numpy()))
            assert np.any(out[0][0])
            assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]), (nu, k)
    for ctx in ctxs:
        ctx.close()


@pytest.mark.parametrize("kw", [dict(smoother=ugmg.SMOOTH_JAC, damp=0.8), dict(), dict(precision=ugmg.MIXED)])
def test_calls_that_do_not_wait(kw, monkeypatch):
    """Alternating levels and columns, more of them than graphs are kept for,
    solves and new parameters in between, with nothing waiting for the GPU:
    no graph goes while it runs."""
    monkeypatch.setenv("UGMG_FUSE_ROWS", "0")     # the lower levels' cycles are replayed too
    P = problems.q1(2, 3, 4, problems.KAPPA_JUMP, seed=2)
    calls = [(4, 1), (4, 3), (4, 1), (4, 3), (4, 0), (4, 1), (3, 2), (4, 3), (3, 2), (3, 1), (4, 1), (3, 1), (2, 3),
             (2, 2), (2, 1), (2, 3), (2, 2), (2, 1), (4, 2), (3, 3), (4, 2), (3, 3), (4, 1), (4, 0)]
    out = []
    for use in (0, 1):
        ctx = ugmg.Context(0)
        ctx.set_stream(torch.cuda.Stream())
        ctx.set_hierarchy(P)
        ctx.set_batch(3)

        def params(nu):
            ctx.set_params(**{**dict(nu1=nu, nu2=nu, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_GS, damp=1.0,
                                     base_abslimit=1e-300, base_maxiter=1, use_graph=use), **kw})

        params(2)
        ctx.preprocess()
        bufs = []
        for k in range(3 * len(calls)):
            level, cols = calls[k % len(calls)]
            f = torch.from_numpy(np.random.default_rng(k).uniform(-1.0, 1.0, (max(cols, 1), P.levels[level].n))).cuda()
            bufs.append((level, cols, torch.zeros_like(f), f))
        xs = torch.zeros(P.levels[-1].n, dtype=torch.float64, device="cuda")
        rhs = torch.from_numpy(P.rhs).cuda()
        torch.cuda.synchronize()
        for k, (level, cols, c, b) in enumerate(bufs):
            if cols != 1:
                ctx.iter_batch(level, c, b)
            else:
                ctx.iter(level, c[0], b[0])
            if k % 17 == 16:
                params(1 + k % 3)
            if k == len(calls):
                ctx.solve(P.top, xs, rhs, red=1e-4, maxiter=5)
        ctx.sync()
        out.append([v.cpu().numpy() for _, _, c, b in bufs for v in (c, b)])
        ctx.close()
    assert all(np.any(v) and np.all(np.isfinite(v)) for v in out[0])
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), k


@pytest.mark.parametrize("kw", [
    dict(smoother=ugmg.SMOOTH_JAC, damp=0.8), dict(smoother=ugmg.SMOOTH_JAC, damp=0.8, nu1=2, nu2=2), dict(),
    dict(precision=ugmg.MIXED)])
def test_local_levels(kw):
    """A cycle on a local level restricts onto the defect that the level below
    holds outside the refined part; a cycle on the level below's list-order
    FP64 vectors before it leaves that alone."""
    P = problems.p1_local(4, 2)
    assert any(np.any(lv.vnclass < 2) for lv in P.levels[3:-1])
    out = []
    for use in (0, 1):
        ctx = ugmg.Context(0)
        ctx.set_stream(torch.cuda.Stream())
        ctx.set_hierarchy(P)
        ctx.set_params(**{**dict(nu1=1, nu2=1, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_GS, damp=1.0,
                                 base_abslimit=1e-300, base_maxiter=1, use_graph=use), **kw})
        ctx.preprocess()
        got = []
        for k in range(3):
            for level in range(2, P.top + 1):
                lv = P.levels[level]
                b = torch.from_numpy(np.random.default_rng(10 * k + level).uniform(-1.0, 1.0, lv.n)).cuda()
                c = torch.zeros_like(b)
                torch.cuda.synchronize()
                ctx.iter(level, c, b)
                ctx.sync()
                got += [c.cpu().numpy(), b.cpu().numpy()]
        ctx.close()
        out.append(got)
    assert all(np.any(v) for v in out[0])
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), k
