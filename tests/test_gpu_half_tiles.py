"""Output-stationary launches of half tiles whose column tiles are wider than their staging rows: results written where nothing is, and
added where something is; whole numbers small enough for every sum to be one."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shape", [(12001, (32, 96)), (12001, (16, 96)), (24000, (24, 72)), (24000, (20, 96))], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_written_and_added(n, shape):
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    vox = clouds.cloud_indoor(clouds.rng_for(5), target=n)
    n = len(vox)
    imap, omap, _, kpos = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    maps = tuple(torch.from_numpy(np.ascontiguousarray(t.astype(np.int32))).cuda() for t in (kpos, imap, omap))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: torch.randint(-1, 2, s, generator=gen, device="cuda").half()
    x, w, start = few(n, shape[0]), few(27, *shape), few(n, shape[1])
    want = exact(x.float(), w.float(), torch.zeros(n, shape[1], device="cuda"), kpos.tolist(), maps[1].long(), maps[2].long())[0]
    assert want.abs().max() <= 2047
    plan = capi.Plan(*maps, n, n)
    out = torch.full((n, shape[1]), float("nan"), device="cuda").half()
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    assert torch.equal(out.double(), want)
    out = start.clone()
    capi.fusion_fwd(x, w, 0, out, maps[0], None, maps[1], maps[2], False, False, plan=plan)
    assert torch.equal(out.double(), want + start.double())
    plan.close()
