"""fp16 output layers of 20 and 28 channels: rows that end in half a 16-byte chunk, over the masked tiles.  Whole numbers
small enough for every sum to be one show a column that went missing or came in from the next row; what lies around every tensor
is NaN."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu


def framed(t):
    """The tensor between NaN, on a 16-byte boundary."""
    room = torch.full((t.numel() + 128,), float("nan"), dtype=t.dtype, device="cuda")
    room[64:64 + t.numel()] = t.reshape(-1)
    return room, room[64:64 + t.numel()].view(t.shape)


# input channels: one, two and three tiles of 32 columns, whole and not; forward slabs of 32, 48 and 64
@pytest.mark.parametrize("n", [130, 3001, 45000])
@pytest.mark.parametrize("shape", [(96, 20), (96, 28), (24, 20), (32, 28), (40, 28), (64, 20), (72, 28), (128, 20), (160, 28)],
                         ids=lambda s: "%dx%d" % s)
def test_whole_numbers(n, shape):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(3), target=n)
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    n = len(vox)
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: torch.randint(0, 40, s, generator=gen, device="cuda").lt(2).half() - torch.randint(0, 40, s, generator=gen, device="cuda").lt(2).half()
    (_, x), (_, w), (_, g) = framed(few(n, shape[0])), framed(few(27, *shape)), framed(few(n, shape[1]))
    want = exact(x.float(), w.float(), g.float(), kpos.tolist(), maps[1].long(), maps[2].long())
    assert max(t.abs().max() for t in want) <= 2048
    around, out = framed(torch.full_like(g, float("nan")))
    plan = capi.Plan(*maps, n, n)
    capi.profile_reset()
    capi.profile_enable(True)
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    gi, gw = torch.full_like(x, float("nan")), torch.full_like(w, float("nan"))
    capi.conv_bwd(g, x, w, gi, gw, *maps, plan=plan)
    capi.profile_enable(False)
    names = [q[0] for q in capi.profile_records()]
    capi.profile_reset()
    assert names == ["gms_rows_kernel(fwd, masked)", "bwd_fused_kernel(masked)"], names
    for got, ref in zip((out, gi, gw), want):
        assert torch.equal(got.double(), ref)
    assert torch.isnan(around[:64]).all() and torch.isnan(around[-64:]).all()
    # added to what is there
    capi.fusion_fwd(x, w, 0, out, maps[0], None, maps[1], maps[2], False, False, plan=plan)
    assert torch.equal(out.double(), 2 * want[0])
    # an infinite row reaches what has a pair with it, and not through the row before it
    rows = torch.tensor([1, n - 1], device="cuda")
    x[rows], g[rows] = float("inf"), float("-inf")
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    capi.conv_bwd(g, torch.zeros_like(x), w, gi, gw, *maps, plan=plan)
    im, om = maps[1].long(), maps[2].long()
    for got, ref, by, to in ((out, want[0], im, om), (gi, want[1], om, im)):
        hit = torch.zeros(n, dtype=torch.bool, device="cuda")
        hit[to[torch.isin(by, rows)]] = True
        assert torch.equal(got[~hit].double(), ref[~hit]) and not torch.isfinite(got[hit]).all()
    plan.close()
