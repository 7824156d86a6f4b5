"""Weight gradients over lists without row bands (no plan, swapped lists): how many slices an offset's pairs are cut into."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def lists(pairs_per_offset, offsets=27, n=20000):
    rng = np.random.default_rng(pairs_per_offset)
    rows = np.concatenate([np.sort(rng.permutation(n)[:pairs_per_offset]) for _ in range(2 * offsets)]).astype(np.int32)
    kpos = np.arange(offsets + 1, dtype=np.int32) * pairs_per_offset
    half = len(rows) // 2
    return tuple(torch.from_numpy(t).cuda() for t in (kpos, rows[:half], rows[half:]))


@pytest.mark.parametrize("c_in,c_out,limit", [(16, 64, 1.25), (16, 16, 1.2)])
def test_a_tenth_more_pairs_take_about_as_long(c_in, c_out, limit):
    """fp16 first layers without a plan, 118 k and 130 k pairs.  (Cut into slices half as long from 124 k pairs on, twice the workgroups
    and twice the atomics, the second took 1.25 to 1.45 times as long.)"""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    n, best = 20000, {}
    x, g = (torch.randint(-1, 2, (n, c), device="cuda").half() for c in (c_in, c_out))
    gw = torch.zeros(27, c_in, c_out, device="cuda").half()
    maps = {m: lists(m) for m in (4380, 4800)}
    for turn in range(8):
        for m, (kpos, im, om) in maps.items():
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(20):
                capi.wgrad(x, g, gw, kpos, im, om)
            stop.record()
            torch.cuda.synchronize()
            best[m] = min(best.get(m, 1e9), start.elapsed_time(stop))
    assert best[4800] < limit * best[4380], best


# pairs on either side of what moves the number of slices: 8 and 27 offsets, tiles wide on either side, and first layers
@pytest.mark.parametrize("shape,dtype", [((64, 128), torch.float16), ((128, 64), torch.float16), ((32, 128), torch.float16), ((128, 32), torch.float16),
                                         ((16, 64), torch.float16), ((16, 64), torch.float32)], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v)[6:])
@pytest.mark.parametrize("offsets,pairs", [(8, 511), (8, 513), (8, 4608), (8, 12288), (8, 18000), (8, 21600), (27, 4608), (27, 6400)])
def test_whole_numbers_on_either_side_of_the_rules(shape, dtype, offsets, pairs):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    n = 24000
    kpos, im, om = lists(pairs, offsets, n)
    few = lambda *s: torch.randint(0, 32, s, device="cuda").lt(1).to(dtype) - torch.randint(0, 32, s, device="cuda").lt(1).to(dtype)
    x, g, w = few(n, shape[0]), few(n, shape[1]), few(offsets, *shape)
    a, b = x.float()[im.long()], g.float()[om.long()]
    want = torch.stack([a[k * pairs:(k + 1) * pairs].T.contiguous() @ b[k * pairs:(k + 1) * pairs] for k in range(offsets)])
    assert want.abs().max() < 2048
    alone, gin, both = torch.zeros_like(w), torch.empty_like(x), torch.full_like(w, float("nan"))
    plan = capi.Plan(kpos, om, im, n, n)
    view = plan.transposed()
    capi.wgrad(x, g, alone, kpos, im, om, plan=view)
    capi.conv_bwd(g, x, w, gin, both, kpos, im, om, plan=view)
    assert torch.equal(alone.float(), want) and torch.equal(both.float(), want)
    view.close()
    plan.close()


# voxels on either side of what leaves a third workgroup on a CU beside 64 x 128 tiles
@pytest.mark.parametrize("shape,n", [((64, 128), 72001), ((64, 128), 85001), ((128, 64), 36001), ((128, 64), 50001), ((128, 64), 62001)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_whole_numbers_beside_the_input_gradient(shape, n):
    from fgms_amd import capi, clouds
    from tests.test_gpu_fp32_parts import exact
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n)
    n = len(vox)
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    few = lambda *s: (torch.randint(0, 32, s, device="cuda").lt(1).float() - torch.randint(0, 32, s, device="cuda").lt(1).float()).half()
    x, g, w = few(n, shape[0]), few(n, shape[1]), few(27, *shape)
    _, want_x, want_w = exact(x, w, g, kpos.tolist(), maps[1].long(), maps[2].long())
    assert max(want_x.abs().max(), want_w.abs().max()) < 2048
    gin, gw = torch.full_like(x, float("nan")), torch.full_like(w, float("nan"))
    plan = capi.Plan(*maps, n, n)
    capi.conv_bwd(g, x, w, gin, gw, *maps, plan=plan)
    assert torch.equal(gin.double(), want_x) and torch.equal(gw.double(), want_w)
    plan.close()
