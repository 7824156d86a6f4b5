"""Whole 128 x 128 weight-gradient tiles dealt to XCDs by their place in the pair lists: every pair counted once, over one
offset, empty ones between others, and the most a plan takes, below and above the size from which the rule applies."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu

FAR = [[900 + i, 900, 900] for i in range(6)]
CUBE, WIDE = clouds.offsets_cube(3).tolist(), clouds.offsets_cube(5).tolist()
OFFSETS = {"one": [[0, 0, 0]], "cube": CUBE, "gaps": FAR[:2] + CUBE[:9] + FAR[2:4] + CUBE[9:] + FAR[4:], "most": WIDE[31:95]}


@pytest.mark.parametrize("offsets", sorted(OFFSETS))
@pytest.mark.parametrize("n,shape", [(4000, (128, 128)), (17000, (128, 128)), (40000, (128, 256))])
def test_against_float64(n, shape, offsets):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(6), target=n)
    offs = np.ascontiguousarray(np.array(OFFSETS[offsets], dtype=np.int32))
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, offs)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda").half()
    x, w, g = draw(len(vox), shape[0]), draw(len(offs), *shape) / 16, draw(len(vox), shape[1]) / 16
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    im, om, kp = maps[1].long(), maps[2].long(), kpos.tolist()
    want, most = exact(x.float(), w.float(), g.float(), kp, im, om)[2], exact(x.float().abs(), w.float().abs(), g.float().abs(), kp, im, om)[2]
    gi, gw = torch.full_like(x, float("nan")), torch.full_like(w, float("nan"))
    capi.conv_bwd(g, x, w, gi, gw, *maps, plan=plan)
    # fp32 sums (a rounding for each 16 products, one for each workgroup of an offset), rounded to fp16 once
    bound = 2.0 ** -11 * want.abs() + 1.1 * (int(knnz.max()) // 16 + 600) * 2.0 ** -24 * most + 2.0 ** -24
    assert ((gw.double() - want).abs() <= bound).all(), ((gw.double() - want).abs() / bound).max()


@pytest.mark.parametrize("n,by_xcd", [(4000, False), (17000, True)])
def test_either_side_of_the_size(n, by_xcd):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(6), target=n)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    x, w, g = (torch.randn(*s, device="cuda").half() for s in ((len(vox), 128), (27, 128, 128), (len(vox), 128)))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    capi.profile_reset()
    capi.profile_enable(True)
    capi.conv_bwd(g, x, w, torch.empty_like(x), torch.empty_like(w), *maps, plan=plan)
    capi.profile_enable(False)
    names = [r[0] for r in capi.profile_records()]
    capi.profile_reset()
    assert ("bwd_fused_kernel(by XCD)" in names) == by_xcd and any(q.startswith("bwd_fused_kernel") for q in names), names


@pytest.mark.parametrize("shape", [(32, 128), (128, 32), (64, 128), (128, 64), (128, 128), (256, 128)], ids=lambda s: "%dx%d" % s)
def test_tiles_of_128_channels_are_exact(shape):
    """Whole numbers small enough for every sum to be one: whatever a stage's rows meet in the wrong place shows.  Lists that
    end inside, at and behind a stage of 64 pairs, both with the input gradient and alone, forward and swapped lists (no bands)."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    sizes = [1, 63, 64, 65, 127, 129, 700, 0, 1500]
    n, rng = 1600, np.random.default_rng(4)
    rows = [np.sort(rng.permutation(n)[:s]) for s in sizes]
    omap = np.concatenate(rows).astype(np.int32)
    imap = np.concatenate([rng.permutation(n)[:s] for s in sizes]).astype(np.int32)
    kpos = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    x, g = (torch.from_numpy(rng.integers(-1, 2, (n, c)).astype(np.float16)).cuda() for c in shape)
    w = torch.from_numpy(rng.integers(-1, 2, (len(sizes), *shape)).astype(np.float16)).cuda()
    for a, b in ((imap, omap), (omap, imap)):
        maps = tuple(torch.from_numpy(t).cuda() for t in (kpos, a, b))
        want = exact(x.float(), w.float(), g.float(), kpos.tolist(), maps[1].long(), maps[2].long())[2]
        assert want.abs().max() < 2048
        plan = capi.Plan(*maps, n, n)
        gi, gw, alone = torch.empty_like(x), torch.full_like(w, float("nan")), torch.zeros_like(w)
        capi.conv_bwd(g, x, w, gi, gw, *maps, plan=plan)
        capi.wgrad(x, g, alone, *maps, plan=plan)
        assert torch.equal(gw.double(), want) and torch.equal(alone.double(), want)
