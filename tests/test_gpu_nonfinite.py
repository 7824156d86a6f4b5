"""Infinities and NaN: a feature or gradient row reaches only what has a pair with it, on every route of
the dispatch, and leaves nothing behind in the library's accumulators.  A weight W[k] reaches every row
with a pair through k; of the rows without one it may turn some into NaN (a zero row times infinity in the
matrix kernels), the others keep their values."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_plan", [True, False], ids=["plan", "no_plan"])
@pytest.mark.parametrize("dtype,tf32", [(np.float16, False), (np.float32, False), (np.float32, True)], ids=["fp16", "fp32", "tf32"])
@pytest.mark.parametrize("n,shape", [(2500, (64, 64)), (2500, (48, 48)), (2500, (24, 40)), (2500, (20, 12)), (2500, (4, 32)), (2500, (96, 128)),
                                     (2500, (128, 256)), (45000, (32, 20)), (45000, (64, 64))])
def test_non_finite_rows_stay_where_they_are(n, shape, dtype, tf32, use_plan):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    rng = np.random.default_rng(n + shape[0])
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=n)
    L = clouds.submanifold_case(vox, *shape, dtype, rng)
    D = G.to_dev(L)
    maps = (D["kpos"], D["imap"], D["omap"])
    plan = capi.Plan(*maps, D["n_in"], D["n_out"]) if use_plan else None
    offset = torch.repeat_interleave(torch.arange(27, device="cuda"), torch.from_numpy(L["knnz"]).cuda().long())
    im, om = D["imap"].long(), D["omap"].long()
    mode = G.mode_of(dtype, tf32)

    def run(x, w, g):
        out, gi, gw = (torch.full_like(t, float("nan")) for t in (g, x, w))
        capi.conv_fwd(x, w, out, *maps, arch80=tf32, plan=plan)
        capi.conv_bwd(g, x, w, gi, gw, *maps, arch80=tf32, plan=plan)
        return out, gi, gw

    def reached(rows, size, by, to):
        hit = torch.zeros(size, dtype=torch.bool, device="cuda")
        mark = torch.zeros(int(max(D["n_in"], D["n_out"])), dtype=torch.bool, device="cuda")
        mark[rows] = True
        hit[to[mark[by]]] = True
        return hit

    def same(got, want, what):
        G.assert_close(got.cpu().numpy(), want.cpu().numpy(), mode, what)

    x, w, g = D["in_feats"], D["kernel"], D["out_grad"]
    clean = run(x, w, g)
    rows = torch.tensor([0, 77, D["n_in"] // 2, D["n_in"] - 1], device="cuda")
    value = torch.tensor([float("inf"), float("nan"), float("-inf"), float("inf")], device="cuda").to(x.dtype)[:, None]

    x2 = x.clone()
    x2[rows] = value
    out, gi, gw = run(x2, w, g)
    hit, hit_k = reached(rows, D["n_out"], im, om), reached(rows, 27, im, offset)
    assert not torch.isfinite(out[hit]).any()
    same(out[~hit], clean[0][~hit], "rows without a pair")
    same(gi, clean[1], "input gradient")
    assert not torch.isfinite(gw[hit_k]).any()
    same(gw[~hit_k], clean[2][~hit_k], "weight gradient")

    g2 = g.clone()
    g2[rows] = value
    out, gi, gw = run(x, w, g2)
    hit, hit_k = reached(rows, D["n_in"], om, im), reached(rows, 27, om, offset)
    assert not torch.isfinite(gi[hit]).any()
    same(gi[~hit], clean[1][~hit], "rows without a pair")
    assert not torch.isfinite(gw[hit_k]).any()
    same(gw[~hit_k], clean[2][~hit_k], "weight gradient")

    k = 5
    w2 = w.clone()
    w2[k] = float("inf")
    out, gi, gw = run(x, w2, g)
    for got, want, to in ((out, clean[0], om), (gi, clean[1], im)):
        hit = torch.zeros(got.shape[0], dtype=torch.bool, device="cuda")
        hit[to[offset == k]] = True
        assert not torch.isfinite(got[hit]).any()
        kept = torch.isfinite(got).all(1)
        assert torch.isnan(got[~hit & ~kept]).all()
        if kept.any():
            same(got[kept], want[kept], "rows the weight did not reach")
    same(gw, clean[2], "weight gradient")

    for got, want in zip(run(x, w, g), clean):            # nothing is left behind
        same(got, want, "clean again")
    if plan is not None:
        plan.close()
