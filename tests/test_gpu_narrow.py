"""Layers with 1 .. 8 (fp16: 16) input channels through a plan: the kernels that stack (offset, channel) pairs
as one contraction.  Sizes around their tiles (32 rows, 64-row blocks, 16 offsets a round, 32 columns), rows at
odd addresses, results added to what a buffer holds -- against the CPU oracle."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def narrow_layer(n_vox, kernel, c_in, c_out, dtype):
    rng = np.random.default_rng(1000 * c_in + n_vox)
    vox = clouds.cloud_planes_spheres(rng, 40 if n_vox < 5000 else 160, max(n_vox, 64))[:n_vox]
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(kernel))
    L = clouds.make_layer(rng, imap, omap, knnz, kpos, len(vox), len(vox), c_in, c_out, dtype)
    return L, G.to_dev(L)


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("n_vox,kernel,c_out", [(1, 3, 32), (33, 3, 8), (65, 3, 64), (1501, 3, 32), (1500, 3, 20), (1501, 5, 40)])
@pytest.mark.parametrize("c_in", [1, 2, 3, 4, 5, 6, 7, 8, 16])
def test_against_oracle(oracle, n_vox, kernel, c_in, c_out, dtype):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    L, D = narrow_layer(n_vox, kernel, c_in, c_out, dtype)
    mode = G.mode_of(L["in_feats"].dtype)
    args = (L["knnz"], L["imap"], L["omap"])
    maps = (D["kpos"], D["imap"], D["omap"])
    plan = capi.Plan(*maps, D["n_in"], D["n_out"])
    ref = oracle.np_fwd(L["in_feats"], L["kernel"], *args, L["n_out"])
    out = torch.full_like(D["out_grad"], float("nan"))
    capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, plan=plan)
    G.assert_close(out.cpu().numpy(), ref, mode, "fwd, written")
    init = torch.randn(D["n_out"], D["c_out"], device="cuda").to(D["in_feats"].dtype)
    G.assert_close(G.run_fwd(capi, D, plan=plan, out_init=init), ref + init.cpu().numpy().astype(np.float64), mode, "fwd, added")
    ref = oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, L["k_vol"])
    for _ in range(2):          # (the second call finds the accumulator as the first one left it)
        gw = torch.full_like(D["kernel"], float("nan"))
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], None, gw, *maps, plan=plan)
        G.assert_close(gw.cpu().numpy(), ref, mode, "wgrad")


@pytest.mark.parametrize("dtype,c_in,c_out", [(np.float16, 4, 64), (np.float32, 4, 64), (np.float32, 8, 32)], ids=["fp16-4", "fp32-4", "fp32-8"])
def test_both_sides_of_the_weight_gradients_rule(oracle, dtype, c_in, c_out):
    """Small launches of shapes that the vector ALUs take as they are stay there; the others, a plan's groups
    of offsets included, go to the matrix cores."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    for n_vox, kernel, want in ((2000, 3, "wgrad_skinny_kernel"), (34000, 3, "wgrad_narrow_kernel"), (9000, 5, "wgrad_narrow_kernel")):
        L, D = narrow_layer(n_vox, kernel, c_in, c_out, dtype)
        maps = (D["kpos"], D["imap"], D["omap"])
        plan = capi.Plan(*maps, D["n_in"], D["n_out"])
        gw = torch.full_like(D["kernel"], float("nan"))
        capi.profile_reset()
        capi.profile_enable(True)
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], None, gw, *maps, plan=plan)
        capi.profile_enable(False)
        names = [r[0] for r in capi.profile_records()]
        capi.profile_reset()
        assert names == [want], (n_vox, names)
        ref = oracle.np_wgrad(L["in_feats"], L["out_grad"], L["knnz"], L["imap"], L["omap"], L["k_vol"])
        G.assert_close(gw.cpu().numpy(), ref, G.mode_of(np.dtype(dtype)), "wgrad %d" % n_vox)


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("c_in", [3, 4, 8])
def test_strided_and_transposed(oracle, c_in, dtype):
    """Two sides of different sizes, and the transposed view of a plan."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    rng = np.random.default_rng(3)
    vox = clouds.cloud_planes_spheres(rng, 40, 1700)
    coarse = np.unique(vox // 2, axis=0).astype(np.int32)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, coarse, clouds.offsets_cube(2), stride=2)
    mode = G.mode_of(np.dtype(dtype))
    for swap in (False, True):
        n_in, n_out = (len(coarse), len(vox)) if swap else (len(vox), len(coarse))
        im, om = (omap, imap) if swap else (imap, omap)
        L = clouds.make_layer(rng, im, om, knnz, kpos, n_in, n_out, c_in, 32, dtype)
        D = G.to_dev(L)
        maps = (D["kpos"], D["imap"], D["omap"])
        plan = (capi.Plan(D["kpos"], D["omap"], D["imap"], n_out, n_in).transposed() if swap
                else capi.Plan(*maps, n_in, n_out))
        args = (knnz, im, om)
        G.assert_close(G.run_fwd(capi, D, plan=plan), oracle.np_fwd(L["in_feats"], L["kernel"], *args, n_out), mode, "fwd")
        gw = torch.zeros_like(D["kernel"])
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], None, gw, *maps, plan=plan)
        G.assert_close(gw.cpu().numpy(), oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, L["k_vol"]), mode, "wgrad")


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("c_in", [3, 8])
def test_non_finite_values_stay_with_their_pairs(oracle, c_in, dtype):
    """An infinite weight or output gradient reaches the rows and offsets that have a pair with it, no others."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    L, D = narrow_layer(1501, 3, c_in, 32, dtype)
    maps = (D["kpos"], D["imap"], D["omap"])
    plan = capi.Plan(*maps, D["n_in"], D["n_out"])
    mode = G.mode_of(np.dtype(dtype))

    def run():
        out, gw = torch.empty_like(D["out_grad"]), torch.empty_like(D["kernel"])
        capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, plan=plan)
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], None, gw, *maps, plan=plan)
        return out, gw

    out0, gw0 = run()
    offset = torch.repeat_interleave(torch.arange(27, device="cuda"), torch.from_numpy(L["knnz"]).cuda().long())
    im, om = D["imap"].long(), D["omap"].long()
    D["kernel"][3] = float("inf")
    out, _ = run()
    hit = torch.zeros(D["n_out"], dtype=torch.bool, device="cuda")
    hit[om[offset == 3]] = True
    assert hit.any() and not hit.all() and not torch.isfinite(out[hit]).any()
    G.assert_close(out[~hit].cpu().numpy(), out0[~hit].cpu().numpy(), mode, "rows without the offset")
    D["kernel"][3] = 0
    D["out_grad"][700] = float("nan")
    _, gw = run()
    hit = torch.zeros(27, dtype=torch.bool, device="cuda")
    hit[offset[om == 700]] = True
    assert hit.any() and not hit.all() and not torch.isfinite(gw[hit]).any()
    G.assert_close(gw[~hit].cpu().numpy(), gw0[~hit].cpu().numpy(), mode, "offsets without the row")
    D["out_grad"][700] = 1
    out, gw = run()
    assert torch.isfinite(out).all() and torch.isfinite(gw).all()       # nothing is left behind
