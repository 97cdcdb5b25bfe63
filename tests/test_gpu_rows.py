"""Row products at the edges of the kernels' chunks: every row width from 1
up past two chunks, uniform-offset and explicit slices, b = 1..4, against
numpy in FP64 (FP32 copies with the FP32 bound)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _level(b, wmax, uniform, seed=0):
    """A diagonally dominant level whose rows have 1..wmax entries: random
    columns, or the offsets +-1, +-2, ... shared by runs of rows."""
    from ug_amd.problems import Level
    rng = np.random.default_rng(seed)
    n = 64 * wmax + 37
    rows = []
    for v in range(n):
        w = 1 + (v // 64 if uniform else v) % wmax
        if uniform:
            offs = [(-1) ** k * (k // 2 + 1) for k in range(w - 1)]
            cols = [v + o for o in offs if 0 <= v + o < n]
        else:
            cols = [int(c) for c in rng.choice(n, w + 1, replace=False) if c != v][:w - 1]
        rows.append([v] + cols)
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    ci = np.concatenate(rows).astype(np.int32)
    vals = rng.uniform(-1.0, 1.0, (len(ci), b, b))
    vals[rp[:-1]] += 4.0 * b * wmax * np.eye(b)
    return Level(n=n, b=b, row_ptr=rp, col_idx=ci, vals=vals.reshape(-1), skip=np.zeros(n, np.uint32),
                 vclass=np.full(n, 3, np.uint8), vnclass=np.zeros(n, np.uint8))


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("b,wmax", [(1, 30), (2, 18), (3, 18), (4, 10)])
def test_row_products(b, wmax, uniform):
    import torch
    from ug_amd import problems, ugmg
    lv = _level(b, wmax, uniform)
    ctx = ugmg.Context(0)
    ctx.set_hierarchy(problems.Problem(dim=1, levels=[lv]))
    ctx.set_params(baselevel=0)
    ctx.preprocess()
    rng = np.random.default_rng(1)
    x = rng.uniform(-1.0, 1.0, (lv.n, b))
    y = rng.uniform(-1.0, 1.0, (lv.n, b))
    blk = lv.vals.reshape(-1, b, b)
    at = np.repeat(np.arange(lv.n), np.diff(lv.row_ptr))
    want, mag = np.zeros((lv.n, b)), np.zeros((lv.n, b))
    np.add.at(want, at, np.einsum("kij,kj->ki", blk, x[lv.col_idx]))
    np.add.at(mag, at, np.einsum("kij,kj->ki", abs(blk), abs(x[lv.col_idx])))
    terms = b * (wmax + 1)
    xt, yt = torch.from_numpy(x.ravel()).cuda(), torch.from_numpy(y.ravel()).cuda()
    torch.cuda.synchronize()
    ctx.dmatmul(0, yt, xt)
    ctx.sync()
    # a sum of `terms` rounded products: at most terms * eps * sum |a x|
    assert np.all(np.abs(yt.cpu().numpy().reshape(-1, b) - want) <= terms * 2.0 ** -52 * mag)
    x32 = torch.from_numpy(x.ravel().astype(np.float32)).cuda()
    y32 = torch.from_numpy(y.ravel().astype(np.float32)).cuda()
    torch.cuda.synchronize()
    ctx.smatmul_minus(0, y32, x32)
    ctx.sync()
    got = y32.cpu().numpy().reshape(-1, b)
    assert np.all(np.abs(got - (y - want)) <= (terms + 3) * 2.0 ** -23 * (mag + abs(y)))
    ctx.close()
