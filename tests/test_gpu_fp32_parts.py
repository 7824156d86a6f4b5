"""fp32 tensors on the 16-bit matrix pipes: three bf16 parts hold a value in full, eight products of parts stand for one.
All three passes against float64, over the grids and tiles of the kernels, for values of either sign, of one
sign, and over many magnitudes; the largest finite numbers stay finite."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from fgms_amd import clouds

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


def errors(values):
    """Errors of a 64 -> 64 layer's three passes against float64: 2-norm relative, and for results that are one product each
    (one weight to a row and column; one output gradient) the root mean square in 2^-24 of the result."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=40000)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    x, w, g = (torch.randn(*s, generator=gen, device="cuda") for s in ((len(vox), 64), (27, 64, 64), (len(vox), 64)))
    if values == "positive":
        x, w, g = x.abs(), w.abs(), g.abs()
    one_w, one_g = torch.zeros_like(w), torch.zeros_like(g)
    one_w[12] = torch.diag(w[12].diagonal())
    one_g[len(vox) // 2] = g[len(vox) // 2]
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    plan = capi.Plan(*maps, len(vox), len(vox))
    im, om, kp = maps[1].long(), maps[2].long(), kpos.tolist()
    found = []
    for weights, gradients, single in ((w, g, False), (one_w, one_g, True)):
        out, gi, gw = (torch.empty_like(t) for t in (g, x, w))
        capi.conv_fwd(x, weights, out, *maps, plan=plan)
        capi.conv_bwd(g, x, weights, gi, gw, *maps, plan=plan)
        if single:
            capi.conv_bwd(gradients, x, w, torch.empty_like(gi), gw, *maps, plan=plan)
        want = exact(x, weights, g, kp, im, om)[:2] + exact(x, w, gradients, kp, im, om)[2:]
        for got, ref in zip((out, gi, gw), want):
            e = got.double() - ref
            if single:
                found.append(2.0 ** 24 * (e[ref != 0] / ref[ref != 0]).square().mean().sqrt().item())
            else:
                found.append((e.norm() / ref.norm()).item())
    return found


@pytest.mark.parametrize("values", ["normal", "positive"])
def test_errors_against_those_of_fp32_mfmas(values):
    """Sums come out closer to the exact ones than those of fp32 MFMAs (FGMS_SPLIT_BF16=0 in a process of its own), which round the
    running sum eight times as often; single products are rounded once on either."""
    code = "import json; from tests.test_gpu_fp32_parts import errors; print('ERRORS ' + json.dumps(errors(%r)))" % values
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, FGMS_SPLIT_BF16="0"), cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    theirs = json.loads([l for l in r.stdout.splitlines() if l.startswith("ERRORS ")][-1][len("ERRORS "):])
    ours = errors(values)
    print(ours, theirs)
    assert all(a <= 0.7 * b for a, b in zip(ours[:2], theirs[:2])), (ours, theirs)
    # (a weight gradient also rounds once for each wave and workgroup, the same on either: at least no worse)
    assert ours[2] <= theirs[2], (ours, theirs)
    # (a sample of 64 x 64 products and more: its root mean square is known to 2 %)
    assert all(a <= 1.05 * b for a, b in zip(ours[3:], theirs[3:])), (ours, theirs)
