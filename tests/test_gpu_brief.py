"""Small fp16 forward launches, whose tiles take all offsets at once: whole numbers small enough for every sum to be one, over the
channel counts and numbers of offsets it takes, first and last rows of a tile, and the plan's forms (a map with its centre kept
apart, a mirrored one, empty offsets, rows without a pair)."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu

BRIEF, HELD = "gms_brief_kernel", "gms_held_kernel"
CUBE, WIDE = clouds.offsets_cube(3).tolist(), clouds.offsets_cube(5).tolist()
OFFSETS = {"cube": CUBE, "17": WIDE[54:71], "32": WIDE[40:72], "gaps": [[900, 900, 900]] + CUBE[:9] + [[901, 900, 900]] + CUBE[9:]}
FEW = {"9": CUBE[9:18], "16": CUBE[5:21], **OFFSETS}


def assert_runs(kernel, call):
    """One launch, and of this kernel; None: neither of the two."""
    from fgms_amd import capi
    capi.profile_reset()
    capi.profile_enable(True)
    call()
    capi.profile_enable(False)
    names = [q for q, _ in capi.profile_records() if q.startswith("gms_")]
    capi.profile_reset()
    assert names == [kernel] if kernel else not {BRIEF, HELD} & set(names), names


@pytest.mark.parametrize("offsets", sorted(OFFSETS))
@pytest.mark.parametrize("n,shape", [(1, (32, 32)), (31, (16, 64)), (33, (48, 32)), (64, (64, 64)), (321, (32, 96)), (2000, (64, 32)), (2047, (32, 32)),
                                     (500, (24, 40)), (700, (56, 16)), (900, (40, 72))],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_whole_numbers(n, shape, offsets):
    whole_numbers(n, shape, offsets, BRIEF)


# up to 32 channels with all weights in LDS: few offsets at any size, more of them above what the other kernel takes; and what neither takes
# (too many channels in or columns, or offsets, for the rows)
@pytest.mark.parametrize("n,shape,offsets", [(1, (32, 32), "9"), (257, (24, 24), "16"), (3001, (32, 16), "9"), (3001, (40, 32), "16"), (40001, (32, 32), "cube"),
                                             (40001, (24, 32), "gaps"), (33000, (32, 24), "32"), (50000, (16, 16), "17"), (1500, (24, 40), "16"),
                                             (3001, (16, 64), "9"), (35000, (32, 64), "cube")])
def test_whole_numbers_with_the_weights_held(n, shape, offsets):
    whole_numbers(n, shape, offsets, None if shape in ((40, 32), (24, 40), (32, 64)) else HELD)


# the rows on either side of each rule: 1 024 tiles of 32 rows and columns in two workgroups a CU, 384 in one; 512 and 1 024 workgroups of 256 rows
# with the weights held
@pytest.mark.parametrize("n,shape,kernel", [(32768, (32, 32), BRIEF), (32769, (32, 32), HELD), (16384, (32, 64), BRIEF), (16385, (32, 64), None),
                                            (12288, (64, 32), BRIEF), (12289, (64, 32), None), (6144, (48, 64), BRIEF), (6145, (48, 64), None),
                                            (131072, (32, 32), HELD), (131073, (32, 32), None), (131073, (32, 16), HELD),
                                            (131072, (16, 64), HELD), (131073, (16, 64), None), (131073, (16, 48), HELD)])
def test_sides_of_the_rules(n, shape, kernel):
    from fgms_amd import capi
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes for 256 CUs")
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n + 4000)[:n]
    assert len(vox) == n
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    x, w = torch.randn(n, shape[0], device="cuda").half(), torch.randn(27, *shape, device="cuda").half()
    out = torch.empty(n, shape[1], device="cuda").half()
    plan = capi.Plan(*maps, n, n)
    assert_runs(kernel, lambda: capi.conv_fwd(x, w, out, *maps, plan=plan))
    plan.close()


@pytest.mark.parametrize("n,kernel", [(114688, HELD), (114689, None)])
def test_sixteen_channels_added_to_64_columns(n, kernel):
    """Results that are added to, of two column tiles a row: up to 896 workgroups of 256 rows."""
    from fgms_amd import capi
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes for 256 CUs")
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n + 4000)[:n]
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    x, w, start = (torch.randint(-2, 3, s, device="cuda").half() for s in ((n, 16), (27, 16, 64), (n, 64)))
    want = exact(x.float(), w.float(), torch.zeros_like(start, dtype=torch.float32), kpos.tolist(), maps[1].long(), maps[2].long())[0]
    plan, out = capi.Plan(*maps, n, n), start.clone()
    assert_runs(kernel, lambda: capi.fusion_fwd(x, w, 0, out, maps[0], None, maps[1], maps[2], False, False, plan=plan))
    assert torch.equal(out.double(), want + start.double())
    plan.close()


def whole_numbers(n, shape, offsets, kernel):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n)
    n = len(vox)
    offs = np.ascontiguousarray(np.array(FEW[offsets], dtype=np.int32))
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, offs)
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: torch.randint(-2, 3, s, generator=gen, device="cuda").half()
    x, w = few(n, shape[0]), few(len(offs), *shape)
    zeros = torch.zeros(n, shape[1], device="cuda")
    want = exact(x.float(), w.float(), zeros, kpos.tolist(), maps[1].long(), maps[2].long())[0]
    assert want.abs().max() <= 2048
    plan = capi.Plan(*maps, n, n)
    out = torch.full_like(zeros, float("nan")).half()
    assert_runs(kernel, lambda: capi.conv_fwd(x, w, out, *maps, plan=plan))
    assert torch.equal(out.double(), want)
    start = few(n, shape[1])
    out = start.clone()
    assert_runs(kernel, lambda: capi.fusion_fwd(x, w, 0, out, maps[0], None, maps[1], maps[2], False, False, plan=plan))
    assert torch.equal(out.double(), want + start.double())
    plan.close()


@pytest.mark.parametrize("n", [95, 2000])
def test_mirrored_plan_and_centre(n):
    from FGMS.nn import KernelMap, sparse_conv
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = torch.from_numpy(clouds.cloud_indoor(clouds.rng_for(4), target=n)).cuda()
    n = len(vox)
    x = torch.randint(-2, 3, (n, 32), device="cuda").half()
    w = torch.randint(-2, 3, (27, 32, 64), device="cuda").half()
    imap, omap, knnz, kpos = capi.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    want = exact(x.float(), w.float(), torch.zeros(n, 64, device="cuda"), kpos.tolist(), imap.long(), omap.long())[0]
    got = []
    with torch.no_grad():
        assert_runs(BRIEF, lambda: got.append(sparse_conv(x, w, KernelMap.from_coords(vox, vox, clouds.offsets_cube(3)), False)))
    assert torch.equal(got[0].double(), want)
    imap, omap, knnz, kpos = capi.build_kernel_map(vox, vox, clouds.offsets_cube(3), skip_offset=13)
    plan = capi.Plan(kpos, imap.clone(), omap.clone(), n, n)
    out = torch.zeros(n, 64, device="cuda").half()
    assert_runs(BRIEF, lambda: capi.fusion_fwd(x, w, 0, out, kpos, None, imap, omap, True, False, plan=plan))
    assert torch.equal(out.double(), want)
    plan.close()


@pytest.mark.parametrize("n,shape", [(1000, (16, 32)), (1000, (32, 64)), (1000, (64, 32)), (40000, (16, 32)), (40000, (32, 24))])
def test_infinite_weights_reach_their_pairs_only(n, shape):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(4), target=n)
    n = len(vox)
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    x, w = torch.randn(n, shape[0], device="cuda").half(), torch.randn(27, *shape, device="cuda").half() / 8
    plan = capi.Plan(*maps, n, n)
    clean, out = (torch.full((n, shape[1]), float("nan"), device="cuda").half() for _ in range(2))
    assert_runs(BRIEF if n == 1000 else HELD, lambda: capi.conv_fwd(x, w, clean, *maps, plan=plan))
    w[5], w[22] = float("inf"), float("nan")
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    hit = torch.zeros(n, dtype=torch.bool, device="cuda")
    for k in (5, 22):
        hit[maps[2][kpos[k]:kpos[k + 1]].long()] = True
    assert hit.any() and not hit.all() and not torch.isfinite(out[hit]).any()
    # (the same products; sums of a few offsets before they meet the others', or of each by itself: fp32 roundings)
    assert torch.allclose(out[~hit].float(), clean[~hit].float(), rtol=2.0 ** -10, atol=2.0 ** -20 * 27 * shape[0])
    plan.close()
