"""fgms_conv_fwd / fgms_conv_bwd write their outputs: buffers full of NaN, rows no pair reaches, one
gradient without the other -- for every kernel family the dispatch has, against the CPU oracle."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def holes(n_side, seed):
    """A map whose last third of output rows and first third of input rows have no pair."""
    rng = np.random.default_rng(seed)
    imap, omap, knnz = [], [], []
    for k in range(27):
        m = 0 if k in (3, 20) else int(rng.integers(1, n_side // 3))
        i = n_side // 3 + rng.permutation(n_side - n_side // 3)[:m]
        o = np.sort(rng.permutation(n_side - n_side // 3)[:m])
        imap.append(i.astype(np.int32)); omap.append(o.astype(np.int32)); knnz.append(m)
    kpos = np.concatenate([[0], np.cumsum(knnz)]).astype(np.int32)
    return np.concatenate(imap), np.concatenate(omap), np.array(knnz, np.int32), kpos


@pytest.mark.parametrize("use_plan", [True, False], ids=["plan", "no_plan"])
@pytest.mark.parametrize("dtype,tf32", [(np.float16, False), (np.float32, False), (np.float32, True)], ids=["fp16", "fp32", "tf32"])
@pytest.mark.parametrize("n,shape", [(65, (32, 32)), (700, (4, 32)), (700, (64, 20)), (1500, (64, 64)), (1500, (16, 16)),
                                     (3000, (32, 256)), (20000, (128, 128)), (70001, (64, 64))])
def test_written_not_added(oracle, n, shape, dtype, tf32, use_plan):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    maps = holes(n, n + shape[0])
    L = clouds.make_layer(np.random.default_rng(7), *maps, n, n, *shape, dtype)
    D = G.to_dev(L)
    mode = G.mode_of(L["in_feats"].dtype, tf32)
    args = (L["knnz"], L["imap"], L["omap"])
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], n, n) if use_plan else None
    nan = lambda *s: torch.full(s, float("nan"), dtype=D["in_feats"].dtype, device="cuda")
    maps = (D["kpos"], D["imap"], D["omap"])
    out = nan(n, shape[1])
    capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, arch80=tf32, plan=plan)
    G.assert_close(out.cpu().numpy(), oracle.c_fwd(L["in_feats"], L["kernel"], *args, n), mode, "fwd")
    ref_gi = oracle.c_dgrad(L["out_grad"], L["kernel"], *args, n)
    ref_gw = oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, 27)
    for want in ((True, True), (True, False), (False, True)):
        gi = nan(n, shape[0]) if want[0] else None
        gw = nan(27, *shape) if want[1] else None
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], gi, gw, *maps, arch80=tf32, plan=plan)
        if want[0]:
            G.assert_close(gi.cpu().numpy(), ref_gi, mode, "dgrad")
        if want[1]:
            G.assert_close(gw.cpu().numpy(), ref_gw, mode, "wgrad")


def test_no_pairs():
    from fgms_amd import capi
    x, w = torch.ones(5, 32, device="cuda"), torch.ones(27, 32, 32, device="cuda")
    kpos = torch.zeros(28, dtype=torch.int32, device="cuda")
    none = torch.zeros(0, dtype=torch.int32, device="cuda")
    out, gi, gw = (torch.full_like(t, 3.0) for t in (x, x, w))
    capi.conv_fwd(x, w, out, kpos, none, none)
    capi.conv_bwd(x, x, w, gi, gw, kpos, none, none)
    assert not out.any() and not gi.any() and not gw.any()


@pytest.mark.parametrize("dtype,tf32", [(np.float16, False), (np.float32, False), (np.float32, True)], ids=["fp16", "fp32", "tf32"])
@pytest.mark.parametrize("n", [1, 127, 129, 16384, 16385, 32768, 32769, 65536, 65537])
def test_small_forward_launches(oracle, n, dtype, tf32):
    """The edges of the choice of column tiles and groups of waves (128-row tiles against 256 CUs)."""
    from fgms_amd import capi
    rng = np.random.default_rng(n)
    knnz = np.array([0 if k == 4 else min(n, 1 + 40 * k) for k in range(27)], np.int32)
    side = lambda: np.concatenate([np.sort(rng.permutation(n)[:m]) for m in knnz]).astype(np.int32)
    kpos = np.concatenate([[0], np.cumsum(knnz)]).astype(np.int32)
    L = clouds.make_layer(rng, side(), side(), knnz, kpos, n, n, 64, 64, dtype)
    D = G.to_dev(L)
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], n, n)
    out = torch.full((n, 64), float("nan"), dtype=D["in_feats"].dtype, device="cuda")
    capi.conv_fwd(D["in_feats"], D["kernel"], out, D["kpos"], D["imap"], D["omap"], arch80=tf32, plan=plan)
    ref = oracle.c_fwd(L["in_feats"], L["kernel"], L["knnz"], L["imap"], L["omap"], n)
    G.assert_close(out.cpu().numpy(), ref, G.mode_of(L["in_feats"].dtype, tf32), "fwd")


@pytest.mark.parametrize("use_plan", [True, False], ids=["plan", "no_plan"])
@pytest.mark.parametrize("dtype,tf32", [(np.float16, False), (np.float32, False), (np.float32, True)], ids=["fp16", "fp32", "tf32"])
@pytest.mark.parametrize("n,shape", [(65, (96, 96)), (900, (48, 96)), (900, (96, 48)), (900, (96, 32)), (900, (32, 96)), (900, (96, 64)),
                                     (900, (64, 96)), (900, (96, 128)), (900, (128, 96)), (900, (24, 96)), (900, (48, 160)), (70001, (96, 96))])
def test_96_and_48_channels(oracle, n, shape, dtype, tf32, use_plan):
    test_written_not_added(oracle, n, shape, dtype, tf32, use_plan)


@pytest.mark.parametrize("n,shape", [(65, (48, 48)), (900, (24, 24)), (900, (16, 32)), (900, (24, 48)), (900, (48, 24)), (900, (40, 56)),
                                     (900, (96, 48)), (900, (80, 72)), (900, (160, 160)), (900, (128, 24)), (900, (104, 136)), (3000, (56, 88)),
                                     (40000, (48, 48)), (70001, (24, 48)), (70001, (48, 160))])
def test_channels_that_fill_no_tile(oracle, n, shape):
    """Masked columns and channels (fp16), at the edges of 16-byte chunks, slabs and 32-column tiles."""
    test_written_not_added(oracle, n, shape, np.float16, False, True)
