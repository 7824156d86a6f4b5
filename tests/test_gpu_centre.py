"""The centre offset kept out of the lists (separate_mid): it rides along in the output-stationary launch where that
kernel serves the pass, and is a product of its own elsewhere -- against the CPU oracle, over the kernel's grids
(groups of waves, shared tiles, the tile table), with a map that lists the centre as well, and with rows that have no other pair."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def centre_layer(n, c_in, c_out, dtype, skip=13):
    rng = np.random.default_rng(n + c_in)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=n + 40)
    vox = np.ascontiguousarray(np.concatenate([vox[:n], vox.max(0) + 9 + 5 * np.arange(1, 70)[:, None] * np.ones((1, 3), int)]).astype(np.int32))
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3), skip_offset=skip)
    L = clouds.make_layer(rng, imap, omap, knnz, kpos, len(vox), len(vox), c_in, c_out, dtype)
    return L, G.to_dev(L)


@pytest.mark.parametrize("dtype,arch80", [(np.float16, False), (np.float32, False), (np.float32, True)], ids=["fp16", "fp32", "tf32"])
@pytest.mark.parametrize("n,shape", [(63, (32, 32)), (1500, (64, 64)), (1500, (48, 96)), (1500, (20, 12)), (1500, (4, 32)), (1500, (128, 256)),
                                     (20000, (32, 32)), (40000, (64, 32)), (70000, (32, 64)), (20000, (24, 48))])
def test_against_oracle(oracle, n, shape, dtype, arch80):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    mode = G.mode_of(np.dtype(dtype), arch80)
    for skip in (13, None) if n == 1500 else (13,):
        L, D = centre_layer(n, *shape, dtype, skip)
        ref = oracle.np_fwd(L["in_feats"], L["kernel"], L["knnz"], L["imap"], L["omap"], L["n_out"], precompute=True)
        init = torch.randn(D["n_out"], D["c_out"], device="cuda").to(D["in_feats"].dtype)
        plan = capi.Plan(D["kpos"], D["imap"], D["omap"], D["n_in"], D["n_out"])
        for p in (plan, None) if n == 1500 else (plan,):
            # the fused call's centre overwrites, the sequential one's is added
            G.assert_close(G.run_fwd(capi, D, True, True, arch80, p, init), ref, mode, "fused")
            G.assert_close(G.run_fwd(capi, D, False, True, arch80, p, init), ref + init.cpu().numpy().astype(np.float64), mode, "sequential")
        plan.close()


# (policy 4: small fp16 layers on the output-stationary kernel too)
@pytest.mark.parametrize("shape,policy,kernel", [((64, 64), 0, "gms_brief_kernel"), ((48, 96), 0, "gms_brief_kernel"), ((64, 64), 4, "gms_rows_kernel(fwd)"),
                                                 ((128, 64), 0, "gms_rows_kernel(fwd)"), ((72, 96), 0, "gms_rows_kernel(fwd, masked)"),
                                                 ((96, 20), 0, "gms_rows_kernel(fwd, masked)")])
def test_one_main_launch(shape, policy, kernel):
    from fgms_amd import capi
    capi.set_kernel_policy(policy)
    L, D = centre_layer(1500, *shape, np.float16)
    plan = capi.Plan(D["kpos"], D["imap"], D["omap"], D["n_in"], D["n_out"])
    G.run_fwd(capi, D, True, True, False, plan)
    capi.profile_reset()
    capi.profile_enable(True)
    G.run_fwd(capi, D, True, True, False, plan)
    capi.profile_enable(False)
    names = [r[0] for r in capi.profile_records()]
    capi.profile_reset()
    plan.close()
    capi.set_kernel_policy(0)
    assert names == [kernel]
