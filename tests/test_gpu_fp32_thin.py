"""fp32 layers over thinned clouds, on either side of the rule between the output-stationary kernel and the pair view:
forward, input gradient alone and both gradients, in fp32 and tf32 mode, against float64, and where the rule sends them."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp32", "tf32"])
@pytest.mark.parametrize("n,full,c,pair_view", [(10000, 40000, 32, {"fp32": True, "tf32": True}), (20000, 60000, 64, {"fp32": True, "tf32": True}),
                                                (60000, 100000, 64, {"fp32": False, "tf32": False}), (60000, 150000, 128, {"fp32": True, "tf32": False}),
                                                (9000, 30000, 256, {"fp32": True, "tf32": True})])
def test_against_float64(n, full, c, pair_view, mode):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=full)
    vox = np.ascontiguousarray(vox[np.sort(np.random.default_rng(1).permutation(len(vox))[:n])])
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x, w, g = draw(n, c), draw(27, c, c), draw(n, c)
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan, tf = capi.Plan(*maps, n, n), mode == "tf32"
    out, gi, gi_alone, gw = (torch.full_like(t, float("nan")) for t in (g, x, x, w))
    capi.profile_reset()
    capi.profile_enable(True)
    capi.conv_fwd(x, w, out, *maps, arch80=tf, plan=plan)
    capi.profile_enable(False)
    assert ("pair view" in capi.profile_records()[0][0]) == pair_view[mode], capi.profile_records()
    capi.conv_bwd(g, x, w, gi, gw, *maps, arch80=tf, plan=plan)
    capi.conv_bwd(g, x, w, gi_alone, None, *maps, arch80=tf, plan=plan)
    im, om, kp = maps[1].long(), maps[2].long(), kpos.tolist()
    want, size = exact(x, w, g, kp, im, om), exact(x.abs(), w.abs(), g.abs(), kp, im, om)
    # a rounding of 2^-24 for each 16 products, and one for each offset's atomic or each of at most 64 workgroups; two
    # parts of 8 bits keep a value to 2^-17: a product of two, and the dropped one, to 2^-16 each
    per_row, per_weight = (27 * c) // 16 + 33, int(knnz.max()) // 16 + 70
    for got, ref, most, roundings in ((out, want[0], size[0], per_row), (gi, want[1], size[1], per_row), (gi_alone, want[1], size[1], per_row), (gw, want[2], size[2], per_weight)):
        bound = (1.1 * roundings * 2.0 ** -24 + (2.0 ** -15 if tf else 0)) * most + 1e-30
        assert ((got.double() - ref).abs() <= bound).all(), ((got.double() - ref).abs() / bound).max()
