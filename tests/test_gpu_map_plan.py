"""Kernel maps from coordinates with their plan in the same pass (KernelMap.from_coords): the lists bit
for bit against the numpy builder, all three passes over the plan against the CPU oracle, at the edges
of the build's blocks, chunks and windows and for every kind of map it tells apart."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def check(oracle, vin, vout, offsets, stride=1, c_in=32, c_out=32, dtype=np.float16, same=True):
    import FGMS.nn as fnn
    rng = np.random.default_rng(len(vin))
    imap, omap, knnz, kpos = clouds.build_kernel_map(vin, vout, offsets, stride)
    L = clouds.make_layer(rng, imap, omap, knnz, kpos, len(vin), len(vout), c_in, c_out, dtype)
    ci = torch.from_numpy(np.ascontiguousarray(vin, np.int32)).cuda()
    co = ci if same else torch.from_numpy(np.ascontiguousarray(vout, np.int32)).cuda()
    kmap = fnn.KernelMap.from_coords(ci, co, offsets, stride)
    for got, want, name in ((kmap.in_map, imap, "in_map"), (kmap.out_map, omap, "out_map"), (kmap.kernel_nnz, knnz, "nnz"),
                            (kmap.kpos, kpos, "kpos")):
        assert np.array_equal(got.cpu().numpy(), want), name
    padded = (knnz.astype(np.int64) + 255) // 256 * 256
    assert np.array_equal(kmap.qkpos.cpu().numpy(), np.concatenate([[0], np.cumsum(padded)])) and kmap.qsum == padded.sum()
    x = torch.from_numpy(L["in_feats"]).cuda().requires_grad_()
    w = torch.from_numpy(L["kernel"]).cuda().requires_grad_()
    y = fnn.sparse_conv(x, w, kmap)
    gx, gw = torch.autograd.grad(y, (x, w), torch.from_numpy(L["out_grad"]).cuda())
    mode, args = G.mode_of(L["in_feats"].dtype), (knnz, imap, omap)
    G.assert_close(y.detach().cpu().numpy(), oracle.c_fwd(L["in_feats"], L["kernel"], *args, len(vout)), mode, "fwd")
    G.assert_close(gx.cpu().numpy(), oracle.c_dgrad(L["out_grad"], L["kernel"], *args, len(vin)), mode, "dgrad")
    G.assert_close(gw.cpu().numpy(), oracle.np_wgrad(L["in_feats"], L["out_grad"], *args, len(offsets)), mode, "wgrad")


def cloud(n, seed=3):
    rng = np.random.default_rng(seed)
    vox = clouds.cloud_indoor(rng, 256, n)
    assert len(vox) == n
    return vox


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 1023, 1025, 2047, 2049, 4097, 66000])
def test_sizes(oracle, n):
    check(oracle, cloud(n), cloud(n), clouds.offsets_cube(3))


@pytest.mark.parametrize("dtype", [np.float16, np.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("shape", [(4, 32), (16, 16), (64, 64), (128, 128), (48, 20)])
def test_shapes_on_a_mirrored_map(oracle, shape, dtype):
    check(oracle, cloud(3000), cloud(3000), clouds.offsets_cube(3), 1, *shape, dtype)


def test_kinds_of_maps(oracle):
    vox = cloud(3001)
    order = np.random.default_rng(1).permutation(len(vox))
    check(oracle, vox[order], vox[order], clouds.offsets_cube(3))                              # rows in no order
    check(oracle, vox * 4 - 300, vox * 4 - 300, clouds.offsets_cube(3) * 4)                   # coordinates a stride apart, negative
    check(oracle, vox, vox, clouds.offsets_cube(3) * 2)                                       # dilated
    check(oracle, vox, vox, clouds.offsets_cube(3)[[1, 0] + list(range(2, 27))])               # offsets that do not mirror
    check(oracle, vox, vox, clouds.offsets_cube(2))                                           # an even kernel
    coarse = clouds.downsample_coords(vox, 2)
    check(oracle, vox, coarse, clouds.offsets_cube(2), 2, 64, 128, same=False)
    check(oracle, vox, coarse, clouds.offsets_cube(3), 2, same=False)                         # overlapping windows
    check(oracle, np.concatenate([vox, vox[::5]]), vox, clouds.offsets_cube(3), same=False)    # repeated input coordinates
    twice = np.concatenate([vox, vox[::5]])
    check(oracle, twice, twice, clouds.offsets_cube(3))                                       # ... on both sides: no mirror image
    check(oracle, vox, vox, clouds.offsets_cube(5), 1, 4, 32)                                 # 125 offsets
    check(oracle, vox[:700], vox[:700], np.concatenate([clouds.offsets_cube(5), clouds.offsets_cube(3) * 4]))   # 152


@pytest.mark.parametrize("k_vol", [1, 8, 9, 33, 41, 63, 64])
def test_numbers_of_offsets(oracle, k_vol):
    """Whole and part bytes of a row's set of offsets, keys of more than 32 bits."""
    check(oracle, cloud(2500), cloud(2500), clouds.offsets_cube(5)[30:30 + k_vol])


def test_sides_of_one_window_and_of_many(oracle):
    vox = cloud(2600)
    coarse = clouds.downsample_coords(vox, 2)
    assert len(coarse) < 1024 < len(vox)
    check(oracle, vox, coarse, clouds.offsets_cube(2), 2, same=False)
    check(oracle, coarse, vox, clouds.offsets_cube(3), 1, same=False)


def test_corners_of_the_coordinate_range():
    """Against the dictionary: the numpy builder's keys of neighbours outside the range meet others'."""
    import FGMS.nn as fnn
    ends = np.array([-(1 << 20), -(1 << 20) + 1, -1, 0, 1, (1 << 20) - 2, (1 << 20) - 1])
    vox = np.stack(np.meshgrid(ends, ends, ends, indexing="ij"), -1).reshape(-1, 3).astype(np.int32)
    offsets, c = clouds.offsets_cube(3), torch.from_numpy(vox).cuda()
    for out, stride in ((vox, 1), (vox // 2, 2)):
        imap, omap, knnz, _ = clouds.build_kernel_map_bruteforce(vox, out, offsets, stride)
        kmap = fnn.KernelMap.from_coords(c, c if stride == 1 else torch.from_numpy(out).cuda(), offsets, stride)
        assert np.array_equal(kmap.in_map.cpu().numpy(), imap) and np.array_equal(kmap.out_map.cpu().numpy(), omap)
        assert np.array_equal(kmap.kernel_nnz.numpy(), knnz)


def test_blocks_of_rows_past_a_thousand():
    """More than 1024 counts to an offset: the lists' prefix sums go round again."""
    import FGMS.nn as fnn
    grid = np.stack(np.meshgrid(np.arange(700), np.arange(400), indexing="ij"), -1).reshape(-1, 2)
    vox = np.concatenate([grid, (grid.sum(1) // 7 % 3)[:, None]], 1).astype(np.int32)
    offsets = clouds.offsets_cube(3)
    imap, omap, knnz, _ = clouds.build_kernel_map(vox, vox, offsets)
    c = torch.from_numpy(vox).cuda()
    kmap = fnn.KernelMap.from_coords(c, c, offsets)
    assert np.array_equal(kmap.in_map.cpu().numpy(), imap) and np.array_equal(kmap.out_map.cpu().numpy(), omap)
    assert np.array_equal(kmap.kernel_nnz.numpy(), knnz)


def test_coordinate_out_of_range():
    import FGMS.nn as fnn
    v = torch.tensor([[0, 0, 0], [1 << 20, 0, 0]], dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError, match="outside"):
        fnn.KernelMap.from_coords(v, v, clouds.offsets_cube(3))


def test_maps_begun_together_and_used_elsewhere(oracle):
    """Several maps begun before the first is used, copies of them, and a first use on another stream."""
    import copy
    import FGMS.nn as fnn
    vox = [cloud(n, n) for n in (900, 2500, 5000)]
    offsets = clouds.offsets_cube(3)
    coords = [torch.from_numpy(v).cuda() for v in vox]
    maps = [fnn.KernelMap.from_coords(c, c, offsets) for c in coords]
    maps.append(copy.copy(maps[0]))
    maps.append(copy.deepcopy(fnn.KernelMap.from_coords(coords[1], coords[1], offsets)))
    dropped = fnn.KernelMap.from_coords(coords[2], coords[2], offsets)
    del dropped
    for m, v in zip(reversed(maps), (vox[1], vox[0], vox[2], vox[1], vox[0])):
        imap, omap, knnz, _ = clouds.build_kernel_map(v, v, offsets)
        x, w = torch.randn(len(v), 32, device="cuda"), torch.randn(27, 32, 32, device="cuda")
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = fnn.sparse_conv(x, w, m)
            im = m.in_map.clone()
        torch.cuda.synchronize()
        assert np.array_equal(im.cpu().numpy(), imap)
        G.assert_close(y.cpu().numpy(), oracle.c_fwd(x.cpu().numpy(), w.cpu().numpy(), knnz, imap, omap, len(v)), "fp32", "fwd")


def test_tiles_of_very_different_weight(oracle):
    """Most voxels alone, the rest in one solid block: equal work per XCD then means very unequal numbers
    of tiles, more than the tile table has room for in one of them."""
    grid = np.stack(np.meshgrid(*[np.arange(38)] * 3, indexing="ij"), -1).reshape(-1, 3)[:50000] * 3
    solid = np.stack(np.meshgrid(*[np.arange(27)] * 3, indexing="ij"), -1).reshape(-1, 3) + [200, 0, 0]
    vox = np.concatenate([grid, solid]).astype(np.int32)
    vox = vox[np.lexsort(vox.T[::-1])]
    vox = np.concatenate([np.zeros((len(vox), cloud(1).shape[1] - 3), np.int32), vox], 1) if cloud(1).shape[1] > 3 else vox
    check(oracle, vox, vox, clouds.offsets_cube(3), 1, 64, 64)


def alone(n, seed=5):
    """Voxels with a block of 2 x 2 x 4 each, an eighth of the blocks of a cube or less: as many searches for a block that is
    there as rows, and most others in vain."""
    rng = np.random.default_rng(seed)
    side = 2 * int(np.ceil(n ** (1 / 3))) + 1
    at = np.sort(rng.choice(side ** 3, n, replace=False))
    return (np.stack([at // side ** 2, at // side % side, at % side], 1) * [2, 2, 4] + rng.integers(0, [2, 2, 4], (n, 3))).astype(np.int32)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 170, 171, 5461, 5462, 20001])
def test_a_block_for_every_row(n):
    """The block table as full as it gets, around sizes that fill its last bucket."""
    import FGMS.nn as fnn
    vox = alone(n)
    c = torch.from_numpy(vox).cuda()
    for offsets in (clouds.offsets_cube(3), clouds.offsets_cube(5)):
        imap, omap, knnz, _ = clouds.build_kernel_map(vox, vox, offsets)
        kmap = fnn.KernelMap.from_coords(c, c, offsets)
        assert np.array_equal(kmap.in_map.cpu().numpy(), imap) and np.array_equal(kmap.out_map.cpu().numpy(), omap)
        assert np.array_equal(kmap.kernel_nnz.numpy(), knnz)


def test_thin_clouds_take_no_longer_at_one_size_than_at_the_next():
    """Just below and just above 4/5 of 2^17 rows with a block each: the larger map is no cheaper.  (With a table of 2^n single slots,
    5/4 a row at least, the smaller one took 6.6 times as long: chains of a hundred dependent probes.)"""
    import FGMS.nn as fnn
    offsets, best = clouds.offsets_cube(5), {}
    coords = {n: torch.from_numpy(alone(n)).cuda() for n in (104000, 106000)}
    for turn in range(6):
        for n, c in coords.items():
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(5):
                fnn.KernelMap.from_coords(c, c, offsets).in_map
            stop.record()
            torch.cuda.synchronize()
            best[n] = min(best.get(n, 1e9), start.elapsed_time(stop))
    assert best[104000] < 2 * best[106000], best
