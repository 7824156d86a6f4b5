"""fp32 channel counts that fill no whole tile, over the kernels that mask the rest: rows shorter than a tile's, at the edges
of row blocks, added to and written, in fp32 and tf32 mode.  Against float64; both modes' bounds from their roundings."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("overwrite", [True, False], ids=["written", "added"])
@pytest.mark.parametrize("mode", ["fp32", "tf32"])
@pytest.mark.parametrize("shape", [(24, 32), (48, 48), (16, 64), (40, 56), (96, 24), (24, 104), (72, 16)])
@pytest.mark.parametrize("n", [65, 9000, 30000])
def test_against_float64(n, shape, mode, overwrite):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + shape[0])
    draw = lambda *s: torch.randn(*s, generator=gen, device="cuda")
    x, w, g = draw(len(vox), shape[0]), draw(27, *shape), draw(len(vox), shape[1])
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    before = [torch.full_like(t, float("nan")) if overwrite else draw(*t.shape) for t in (g, x, w)]
    # (64 values more behind each result: nothing past the end may change)
    flat = [torch.full((t.numel() + 64,), 7.0, device="cuda") for t in before]
    out, gi, gw = (f[:t.numel()].view(t.shape).copy_(t) for f, t in zip(flat, before))
    tf = mode == "tf32"
    if overwrite:
        capi.conv_fwd(x, w, out, *maps, arch80=tf, plan=plan)
        capi.conv_bwd(g, x, w, gi, gw, *maps, arch80=tf, plan=plan)
    else:
        capi.fusion_fwd(x, w, 0, out, maps[0], None, *maps[1:], False, tf, plan=plan)
        capi.bwd(g, x, w, 0, gi, gw, maps[0], None, *maps[1:], False, tf, plan=plan)
    im, om, kp = maps[1].long(), maps[2].long(), kpos.tolist()
    want, size = exact(x, w, g, kp, im, om), exact(x.abs(), w.abs(), g.abs(), kp, im, om)
    # A result is a sum of its products' roundings (one for each 16 products, each tile added by at most 64 workgroups, the
    # value added to) of 2^-24; two parts of 8 bits keep a value to 2^-17, so a product of two to 2^-16 and the dropped one to 2^-16.
    steps = ((27 * shape[0] + 15) // 16 + 6, (27 * shape[1] + 15) // 16 + 6, int(knnz.max()) // 16 + 70)
    for got, was, ref, most, roundings, f in zip((out, gi, gw), before, want, size, steps, flat):
        if not overwrite:
            ref, most = ref + was.double(), most + was.double().abs()
        bound = (1.1 * roundings * 2.0 ** -24 + (2.0 ** -15 if tf else 0)) * most + 1e-30
        assert ((got.double() - ref).abs() <= bound).all(), ((got.double() - ref).abs() / bound).max()
        assert (f[got.numel():] == 7.0).all()


@pytest.mark.parametrize("mode", ["fp32", "tf32"])
@pytest.mark.parametrize("n,shape,masked", [(30000, (48, 48), True), (30000, (40, 56), True), (30000, (64, 64), False)])
def test_which_kernels_run(n, shape, masked, mode):
    """Dense maps and such counts go to the masked tiles, in both passes; whole tiles do not."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    x, w, g = (torch.randn(*s, device="cuda") for s in ((len(vox), shape[0]), (27, *shape), (len(vox), shape[1])))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    capi.profile_reset()
    capi.profile_enable(True)
    capi.conv_fwd(x, w, torch.empty_like(g), *maps, arch80=mode == "tf32", plan=plan)
    capi.conv_bwd(g, x, w, torch.empty_like(x), torch.empty_like(w), *maps, arch80=mode == "tf32", plan=plan)
    capi.profile_enable(False)
    names = [r[0] for r in capi.profile_records()]
    capi.profile_reset()
    assert [q.split("(")[0] for q in names] == ["gms_rows_kernel", "bwd_fused_kernel"], names
    assert [("masked" in q, "bf16x3" in q) for q in names] == [(masked, mode == "tf32")] * 2, names
