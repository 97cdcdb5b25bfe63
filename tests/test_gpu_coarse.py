"""Coarse levels in one workgroup per column (k_coarse_down, k_coarse_up)
against a launch per operation (UGMG_FUSE_ROWS=0): the same bits, for both
smoothers and precisions, several columns, step counts, c += (the second
cycle of a mixed step), levels at and past the limit, local levels whose
coarse vectors keep their value in the restriction, and a finest level smaller
than the one below it."""
import dataclasses

import numpy as np
import pytest

from ug_amd import problems, ugmg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _patch(dim, cells, nref, m):
    """A level that holds the refined elements alone: q1's levels and on top
    the m^dim fine nodes at the origin, the coarse vectors outside keep their
    defect (VNCLASS 0)."""
    F = problems.q1(dim, cells, nref + 1, problems.KAPPA_JUMP, seed=9)
    fine, coarse = F.levels[-1], F.levels[-2]

    def inside(lv, k):
        at = np.arange(lv.n)
        return np.all([at // lv.nodes_per_dir ** d % lv.nodes_per_dir < k for d in range(dim)], axis=0)

    keep = np.flatnonzero(inside(fine, m))
    rim = ~inside(fine, m - 1)                    # zero corrections, identity rows
    new = np.full(fine.n, -1)
    new[keep] = np.arange(keep.size)
    rp, ci, va, pp, pi, pw = [0], [], [], [0], [], []
    for v in keep:
        for q in range(fine.row_ptr[v], fine.row_ptr[v + 1]):
            w = fine.col_idx[q]
            if w == v or (not rim[v] and new[w] >= 0):
                ci.append(new[w])
                va.append(1.0 if rim[v] else fine.vals[q])
        rp.append(len(ci))
        for q in range(fine.p_ptr[v], fine.p_ptr[v + 1]):
            pi.append(fine.p_idx[q])
            pw.append(fine.p_w[q])
        pp.append(len(pi))
    top = dataclasses.replace(
        fine, n=keep.size, row_ptr=np.array(rp, np.int32), col_idx=np.array(ci, np.int32), vals=np.array(va),
        skip=(fine.skip | rim).astype(fine.skip.dtype)[keep], vclass=fine.vclass[keep], vnclass=fine.vnclass[keep],
        nodes_per_dir=m, p_ptr=np.array(pp, np.int32), p_idx=np.array(pi, np.int32), p_w=np.array(pw))
    under = np.where(inside(coarse, m // 2 + 1), 3, 0).astype(coarse.vnclass.dtype)
    F.levels[-2:] = [dataclasses.replace(coarse, vnclass=under), top]
    return F


def _cycle(P, monkeypatch, rows, cols=1, cycles=1, **kw):
    if rows is None:
        monkeypatch.delenv("UGMG_FUSE_ROWS", raising=False)
    else:
        monkeypatch.setenv("UGMG_FUSE_ROWS", str(rows))
    lv = P.levels[-1]
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(P)
    prm = dict(nu1=2, nu2=2, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_GS, damp=1.0, base_abslimit=1e-300,
               base_maxiter=1)
    prm.update(kw)
    ctx.set_params(**prm)
    if cols > 1:
        ctx.set_batch(cols)
    ctx.preprocess()
    b = torch.from_numpy(np.random.default_rng(3).uniform(-1.0, 1.0, (cols, lv.n))).cuda()
    b[:, torch.from_numpy(lv.skip & 1 == 1).cuda()] = 0.0
    c = torch.zeros_like(b)
    torch.cuda.synchronize()
    for _ in range(cycles):
        if cols > 1:
            ctx.iter_batch(P.top, c, b)
        else:
            ctx.iter(P.top, c[0], b[0])
    ctx.sync()
    ctx.close()
    return c.cpu().numpy(), b.cpu().numpy()


def _poison(P, precision, cols=1024):
    """Cycles on NaN in more workgroups than there are CUs."""
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(P)
    ctx.set_params(nu1=1, nu2=1, gamma=1, baselevel=1, smoother=ugmg.SMOOTH_GS, damp=1.0, base_abslimit=1e-300,
                   base_maxiter=1, precision=precision)
    ctx.set_batch(cols)
    ctx.preprocess()
    b = torch.full((cols, P.levels[-1].n), float("nan"), dtype=torch.float64, device="cuda")
    c = torch.zeros_like(b)
    torch.cuda.synchronize()
    ctx.iter_batch(P.top, c, b)
    ctx.sync()
    ctx.close()


CASES = [
    ("2d", lambda: problems.q1(2, 3, 5, problems.KAPPA_JUMP, seed=1), dict(smoother=ugmg.SMOOTH_JAC, damp=0.8, nu1=1, nu2=3)),
    ("2d", lambda: problems.q1(2, 2, 5, problems.KAPPA_ONE, seed=2), dict(baselevel=0, damp=0.9, precision=ugmg.MIXED)),
    ("3d", lambda: problems.q1(3, 1, 5, problems.KAPPA_JUMP, seed=3), dict(nu1=0, nu2=2)),
    ("3d", lambda: problems.q1(3, 3, 3, problems.KAPPA_JUMP, seed=4), dict(baselevel=2, nu1=3, nu2=1, precision=ugmg.MIXED,
                                                                          inner_cycles=2)),
    ("3d cols", lambda: problems.q1(3, 1, 4, problems.KAPPA_JUMP, seed=5), dict(cols=3)),
    ("3d jac", lambda: problems.q1(3, 1, 4, problems.KAPPA_JUMP, seed=6), dict(smoother=ugmg.SMOOTH_JAC, damp=0.8, cols=2,
                                                                              nu2=0)),
    ("3d below", lambda: problems.q1(3, 1, 5, problems.KAPPA_JUMP, seed=8), dict(precision=ugmg.MIXED, inner_cycles=2,
                                                                                cycles=3)),
    ("p1", lambda: problems.p1_cd(5, 1e-3, float("nan"), seed=7), dict(cycles=2)),
    ("local", lambda: problems.p1_local(3, 3), dict(cycles=2)),
    ("local jac", lambda: problems.p1_local(4, 2), dict(smoother=ugmg.SMOOTH_JAC, damp=0.8, cycles=2)),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_coarse_levels_are_bitwise_the_separate_launches(k, monkeypatch):
    tag, make, kw = CASES[k]
    P = make()
    print(f"coarse {k} {tag} {[lv.n for lv in P.levels]}", flush=True)
    want = _cycle(P, monkeypatch, 0, **kw)
    assert np.all(np.isfinite(want[0])) and np.any(want[0])
    for rows in (None, P.levels[-2].n, P.levels[-2].n - 1):
        got = _cycle(P, monkeypatch, rows, **kw)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), rows


@pytest.mark.parametrize("dim,cells,nref,m", [(2, 2, 4, 19), (3, 1, 3, 7)])
@pytest.mark.parametrize("precision", [ugmg.FP64, ugmg.MIXED])
def test_finest_level_smaller_than_the_one_below(dim, cells, nref, m, precision, monkeypatch):
    """The sweeps of a level with more vectors than the finest one start from
    zeros, whatever the workgroup's memory held (here NaN, on every CU)."""
    P = _patch(dim, cells, nref, m)
    print(f"patch {[lv.n for lv in P.levels]}", flush=True)
    assert P.levels[-1].n < P.levels[-2].n <= 1200
    want = _cycle(P, monkeypatch, 0, cycles=2, precision=precision)
    assert np.all(np.isfinite(want[0])) and np.any(want[0])
    below = dataclasses.replace(P, levels=P.levels[:-1])
    for cols in (1, 3):
        monkeypatch.delenv("UGMG_FUSE_ROWS", raising=False)
        _poison(below, precision)
        got = _cycle(P, monkeypatch, None, cols=cols, cycles=2, precision=precision)
        if cols == 1:
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert np.all(np.isfinite(got[0])) and np.all(np.isfinite(got[1]))


@pytest.mark.parametrize("smoother,damp", [(ugmg.SMOOTH_JAC, 0.8), (ugmg.SMOOTH_GS, 1.0)])
def test_surface_solve_is_bitwise_the_separate_launches(smoother, damp, monkeypatch):
    """Every level's correction is there after a cycle: the surface solve adds
    them into x level by level."""
    P = problems.p1_local(4, 2)
    fs = problems.surface_rhs(P, 1, 4)
    out = []
    for rows in (0, 12288):
        monkeypatch.setenv("UGMG_FUSE_ROWS", str(rows))
        ctx = ugmg.Context(0)
        ctx.set_hierarchy(P)
        ctx.set_params(nu1=2, nu2=2, gamma=1, baselevel=1, smoother=smoother, damp=damp, base_abslimit=1e-300,
                       base_maxiter=1)
        ctx.preprocess()
        out.append(ctx.solve_surface_host(P.top, fs, red=1e-8, maxiter=30))
        ctx.close()
    (x0, b0, r0, _), (x1, b1, r1, _) = out
    assert r0.number_of_linear_iterations == r1.number_of_linear_iterations
    for l in range(1, P.top + 1):
        assert np.array_equal(x0[l], x1[l]) and np.array_equal(b0[l], b1[l]), l
