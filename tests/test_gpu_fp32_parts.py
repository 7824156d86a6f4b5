"""fp32 tensors on the 16-bit matrix pipes: three bf16 parts hold a value in full, six products of parts stand for one.
All three passes against float64, over the grids and tiles of the kernels, for values of either sign, of one
sign, and over many magnitudes; the largest finite numbers stay finite."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds

pytestmark = pytest.mark.gpu


def exact(x, w, g, kpos, im, om):
    y, gx, gw = (torch.zeros(n, c, dtype=torch.float64, device="cuda") for n, c in ((g.shape[0], w.shape[2]), (x.shape[0], w.shape[1]), (1, 1)))
    gw = torch.zeros(w.shape, dtype=torch.float64, device="cuda")
    for k in range(w.shape[0]):
        a, b = kpos[k], kpos[k + 1]
        if b > a:
            xi, gi = x[im[a:b]].double(), g[om[a:b]].double()
            y.index_add_(0, om[a:b], xi @ w[k].double())
            gx.index_add_(0, im[a:b], gi @ w[k].double().t().contiguous())
            gw[k] = xi.t().contiguous() @ gi
    return y, gx, gw


@pytest.mark.parametrize("values", ["normal", "positive", "wide"])
@pytest.mark.parametrize("n,shape,thin", [(65, (32, 32), False), (1500, (64, 64), False), (1500, (96, 160), False), (9000, (32, 64), False),
                                          (9000, (256, 128), True), (30000, (64, 32), False), (70000, (64, 64), False)])
def test_against_float64(n, shape, thin, values):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    rng = np.random.default_rng(n)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=4 * n if thin else n)
    if thin:
        vox = np.ascontiguousarray(vox[np.sort(rng.permutation(len(vox))[:n])])
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)

    def draw(*s):
        v = torch.randn(*s, generator=gen, device="cuda")
        return v if values == "normal" else v.abs() if values == "positive" else torch.exp(3 * v) * torch.randn(*s, generator=gen, device="cuda").sign()

    x, w, g = draw(len(vox), shape[0]), draw(27, *shape), draw(len(vox), shape[1])
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    out, gi, gw = (torch.full_like(t, float("nan")) for t in (g, x, w))
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    capi.conv_bwd(g, x, w, gi, gw, *maps, plan=plan)
    im, om, kp = maps[1].long(), maps[2].long(), kpos.tolist()
    want, size = exact(x, w, g, kp, im, om), exact(x.abs(), w.abs(), g.abs(), kp, im, om)
    # Every 16 products round the running sum once, and the small parts' sum, 2^-7 of it, six times as often; a tile is
    # added up by at most 64 workgroups: |error| <= roundings x 2^-24 x the sum of the products' sizes.
    steps = ((27 * shape[0] + 15) // 16 + 4, (27 * shape[1] + 15) // 16 + 4, int(knnz.max()) // 16 + 68)
    for got, ref, most, roundings, what in zip((out, gi, gw), want, size, steps, ("fwd", "dgrad", "wgrad")):
        bound = 1.1 * roundings * 2.0 ** -24 * most + 1e-30
        assert ((got.double() - ref).abs() <= bound).all(), (what, ((got.double() - ref).abs() / bound).max())
        # ... and they are of either sign: the square root of their number, each at most half a unit
        rel = ((got.double() - ref).norm() / ref.norm()).item()
        if values != "wide":
            assert rel <= 2.0 ** -24 * max(2.0, roundings ** 0.5), (what, rel)


def test_large_values_stay_finite():
    """The upper part of a value is cut off, not rounded: the largest finite number does not become infinite."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_planes_spheres(np.random.default_rng(3), 40, 900)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    top = torch.finfo(torch.float32).max
    x = torch.zeros(len(vox), 32, device="cuda")
    x[:, 3] = top
    w = torch.zeros(27, 32, 32, device="cuda")
    w[13] = torch.eye(32, device="cuda") * 0.5
    out = torch.empty(len(vox), 32, device="cuda")
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    assert torch.equal(out, x * 0.5)
