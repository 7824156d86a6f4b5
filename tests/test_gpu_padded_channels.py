"""Channel counts that no tuned kernel takes: one off the kernels' multiples on either side, one
channel, a kernel of more than 64 offsets, with and without a plan, results added to what the
buffers hold -- against the CPU oracle.  fp16 runs over padded copies (or masked), small fp32 calls on
the vector ALUs, bigger ones over copies: the last tests stand on both sides of that rule."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G
from tests.test_gpu_parity import layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_plan", [True, False], ids=["plan", "no_plan"])
@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1), (3, 32), (5, 17), (16, 65), (17, 16), (31, 33), (33, 31), (95, 20), (127, 129)])
def test_against_oracle(oracle, shape, dtype, use_plan):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    L = layer(400 + shape[0], *shape, dtype)
    D = G.to_dev(L)
    mode = G.mode_of(L["in_feats"].dtype)
    args = (L["knnz"], L["imap"], L["omap"])
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], D["n_in"], D["n_out"]) if use_plan else None
    init = torch.randn(D["n_out"], D["c_out"], device="cuda").to(D["in_feats"].dtype)
    ref = oracle.np_fwd(L["in_feats"], L["kernel"], *args, L["n_out"]) + init.cpu().numpy().astype(np.float64)
    G.assert_close(G.run_fwd(capi, D, plan=plan, out_init=init), ref, mode, "fwd")
    for split in (False, True):
        gi, gw = G.run_bwd(capi, D, plan=plan, split=split)
        G.assert_close(gi, oracle.np_dgrad(L["out_grad"], L["kernel"], *args, L["n_in"]), mode, "dgrad")
        G.assert_close(gw, oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, L["k_vol"]), mode, "wgrad")


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("c_in", [3, 4])
def test_wide_kernel(oracle, dtype, c_in):
    """125 offsets: the copies are made once, the offset groups run over them."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    rng = np.random.default_rng(5)
    vox = clouds.cloud_planes_spheres(rng, 40, 1501)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(5))
    L = clouds.make_layer(rng, imap, omap, knnz, kpos, len(vox), len(vox), c_in, 32, dtype)
    D = G.to_dev(L)
    mode = G.mode_of(L["in_feats"].dtype)
    args = (L["knnz"], L["imap"], L["omap"])
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], D["n_in"], D["n_out"])
    G.assert_close(G.run_fwd(capi, D, plan=plan), oracle.np_fwd(L["in_feats"], L["kernel"], *args, L["n_out"]), mode, "fwd")
    gi, gw = G.run_bwd(capi, D, plan=plan)
    G.assert_close(gi, oracle.np_dgrad(L["out_grad"], L["kernel"], *args, L["n_in"]), mode, "dgrad")
    G.assert_close(gw, oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, L["k_vol"]), mode, "wgrad")


def cloud_layer(n_vox, c_in, c_out, dtype, thin=False):
    rng = np.random.default_rng(n_vox + c_in)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=4 * n_vox if thin else n_vox)
    if thin:
        vox = np.ascontiguousarray(vox[np.sort(rng.permutation(len(vox))[:n_vox])])
    return clouds.submanifold_case(vox, c_in, c_out, dtype, rng)


@pytest.mark.parametrize("tf32", [False, True], ids=["fp32", "tf32"])
@pytest.mark.parametrize("shape", [(32, 20), (24, 24), (48, 48), (5, 32), (17, 33)])
def test_fp32_side_of_the_rule(oracle, shape, tf32):
    """Small fp32 calls run on the vector ALUs without copies, bigger ones over copies on the matrix cores, and a thin
    map's weight gradient by its own rule; all of them against the oracle."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    for n, thin in ((1500, False), (45000, False), (40000, True)):
        L = cloud_layer(n, *shape, np.float32, thin)
        D = G.to_dev(L)
        maps = (D["kpos"], D["imap"], D["omap"])
        plan = capi.Plan(*maps, D["n_in"], D["n_out"])
        out, gi, gw = (torch.full_like(t, float("nan")) for t in (D["out_grad"], D["in_feats"], D["kernel"]))
        names = {}
        for what, call in (("fwd", lambda: capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, arch80=tf32, plan=plan)),
                           ("dgrad", lambda: capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], gi, None, *maps, arch80=tf32, plan=plan)),
                           ("wgrad", lambda: capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], None, gw, *maps, arch80=tf32, plan=plan))):
            capi.profile_reset()
            capi.profile_enable(True)
            call()
            capi.profile_enable(False)
            names[what] = [r[0] for r in capi.profile_records()]
        capi.profile_reset()
        if n == 1500:
            assert names["fwd"] == ["generic_gms_kernel(fwd)"] and names["dgrad"] == ["generic_gms_kernel(dgrad)"]
        elif not thin:
            assert not any("generic" in k for ks in names.values() for k in ks)
        elif shape == (48, 48):
            assert names["wgrad"] == ["generic_wgrad_kernel"]
        args = (L["knnz"], L["imap"], L["omap"])
        ref = (oracle.c_fwd(L["in_feats"], L["kernel"], *args, L["n_out"]), oracle.c_dgrad(L["out_grad"], L["kernel"], *args, L["n_in"]),
               oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, L["k_vol"]))
        both = torch.full_like(gi, float("nan")), torch.full_like(gw, float("nan"))
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], *both, *maps, arch80=tf32, plan=plan)
        mode = G.mode_of(np.float32, tf32)
        for got, want, what in zip((out, gi, gw) + both, ref + ref[1:], ("fwd", "dgrad", "wgrad", "dgrad of both", "wgrad of both")):
            G.assert_close(got.cpu().numpy(), want, mode, "%s %d" % (what, n))
        plan.close()


@pytest.mark.parametrize("c_in", [3, 5])
def test_wide_kernel_fp32_over_copies(oracle, c_in):
    """125 offsets over a cloud big enough for the copies: one copy, two groups of offsets."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    rng = np.random.default_rng(6)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=20000)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(5))
    L = clouds.make_layer(rng, imap, omap, knnz, kpos, len(vox), len(vox), c_in, 32, np.float32)
    D = G.to_dev(L)
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], D["n_in"], D["n_out"])
    init = torch.randn(D["n_out"], 32, device="cuda")
    G.run_fwd(capi, D, plan=plan)
    capi.profile_reset()
    capi.profile_enable(True)
    out = G.run_fwd(capi, D, plan=plan, out_init=init)
    capi.profile_enable(False)
    names = [r[0] for r in capi.profile_records()]
    capi.profile_reset()
    assert len(names) == 2 and not any("generic" in n for n in names), names
    G.assert_close(out - init.cpu().numpy(), oracle.c_fwd(L["in_feats"], L["kernel"], L["knnz"], L["imap"], L["omap"], L["n_out"]), "fp32", "fwd")
