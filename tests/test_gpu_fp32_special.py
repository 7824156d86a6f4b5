"""fp32 layers in full precision where values leave the ordinary range: what an infinite value reaches is what fp32
arithmetic makes of it, by sign, on every route, and the rest keeps its values."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu

# Tiles of 32 and 64 columns, with one, two and four groups of waves, 256-row tiles, a table of tiles, the pair view (thinned), channel
# counts that fill no whole tile, and no plan at all
CASES = [(65, (32, 32), "dense"), (1500, (64, 64), "dense"), (9000, (32, 64), "dense"), (9000, (64, 64), "dense"), (30000, (64, 32), "dense"),
         (70000, (64, 64), "dense"), (9000, (96, 160), "dense"), (9000, (256, 128), "thin"), (9000, (48, 48), "dense"), (30000, (40, 56), "dense"),
         (9000, (24, 104), "dense"), (3000, (64, 64), "no plan")]


class Layer:
    """A layer over a cloud: maps, plan, values, and its three passes -- both gradients in one call and each in its own."""

    def __init__(self, n, shape, cloud):
        from fgms_amd import capi
        capi.set_kernel_policy(0)
        vox = clouds.cloud_indoor(clouds.rng_for(2), target=4 * n if cloud == "thin" else n)
        if cloud == "thin":
            vox = np.ascontiguousarray(vox[np.sort(np.random.default_rng(n).permutation(len(vox))[:n])])
        imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
        self.n, self.shape, self.capi, self.most = len(vox), shape, capi, int(knnz.max())
        self.maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
        self.kpos, self.im, self.om = kpos.tolist(), self.maps[1].long(), self.maps[2].long()
        self.offset = torch.repeat_interleave(torch.arange(27, device="cuda"), torch.from_numpy(knnz).cuda().long())
        self.plan = None if cloud == "no plan" else capi.Plan(*self.maps, self.n, self.n)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(n + shape[0])
        self.values = tuple(torch.randn(*s, generator=gen, device="cuda") for s in ((self.n, shape[0]), (27, *shape), (self.n, shape[1])))

    def run(self, x, w, g):
        """(name, result, which of exact()'s results it is)"""
        new = lambda t: torch.full_like(t, float("nan"))
        out, gi, gi_alone, gw, gw_alone = new(g), new(x), new(x), new(w), new(w)
        self.capi.conv_fwd(x, w, out, *self.maps, plan=self.plan)
        self.capi.conv_bwd(g, x, w, gi, gw, *self.maps, plan=self.plan)
        self.capi.conv_bwd(g, x, w, gi_alone, None, *self.maps, plan=self.plan)
        self.capi.conv_bwd(g, x, w, None, gw_alone, *self.maps, plan=self.plan)
        return (("fwd", out, 0), ("dgrad", gi, 1), ("dgrad alone", gi_alone, 1), ("wgrad", gw, 2), ("wgrad alone", gw_alone, 2))

    def exact(self, x, w, g):
        return exact(x, w, g, self.kpos, self.im, self.om)

    def bounds(self, x, w, g):
        """Every addition and every product rounds by 2^-24 of what has been summed up by then, in sizes."""
        terms = (27 * self.shape[0] + 64, 27 * self.shape[1] + 64, self.most + 64)
        return [n * 2.0 ** -24 * t for n, t in zip(terms, self.exact(x.abs(), w.abs(), g.abs()))]


def same_where_beyond(got, want, allowed, what):
    """Infinities and NaN are where they have to be, and nothing else is."""
    beyond = ~torch.isfinite(want)
    assert beyond.any(), what
    assert torch.equal(torch.nan_to_num(got[beyond], nan=7.0), torch.nan_to_num(want[beyond].float(), nan=7.0)), what
    rest = torch.where(beyond, torch.zeros_like(want), (got.double() - want).abs())
    assert (rest <= torch.where(beyond, torch.zeros_like(want), allowed)).all(), what


@pytest.mark.parametrize("n,shape,cloud", CASES)
def test_infinities_keep_their_sign(n, shape, cloud):
    layer = Layer(n, shape, cloud)
    x, w, g = layer.values
    bounds = layer.bounds(x, w, g)
    rows = [0, n // 3, layer.n // 2 + 1, layer.n - 1]
    for t, results in ((x, (0, 2)), (g, (1, 2))):
        t = t.clone()
        for i, (r, v) in enumerate(zip(rows, (float("inf"), float("-inf"), float("inf"), float("nan")))):
            t[r, (7 * i + 3) % t.shape[1]] = v
        values = (t, w, g) if results[0] == 0 else (x, w, t)
        want = layer.exact(*values)
        for what, got, i in layer.run(*values):
            if i in results:
                same_where_beyond(got, want[i], bounds[i], what)
            else:
                assert ((got.double() - want[i]).abs() <= bounds[i]).all(), what

    # One infinite weight: the rows with a pair through its offset get it by sign in its column; a row without one may turn into NaN
    # there (no neighbour, as zeros, times infinity), or keeps its value.
    w2 = w.clone()
    k = int(torch.bincount(layer.offset[layer.offset != 13], minlength=27).argmax())
    w2[k, 3, 7] = float("inf")
    want, clean = layer.exact(x, w2, g), layer.exact(x, w, g)
    for what, got, i in layer.run(x, w2, g):
        if i == 2:
            assert ((got.double() - clean[2]).abs() <= bounds[2]).all(), what
            continue
        beyond = ~torch.isfinite(want[i])
        assert beyond.any() and torch.equal(got[beyond], want[i][beyond].float()), what
        turned = torch.isnan(got) & ~beyond
        column = torch.zeros_like(turned)
        column[:, 7 if i == 0 else 3] = True
        assert not (turned & ~column).any(), what
        kept = ~beyond & ~turned
        assert ((got.double() - clean[i]).abs()[kept] <= bounds[i][kept]).all(), what
