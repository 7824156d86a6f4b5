"""Thin maps one of whose offsets meets every destination row once: its products are written first, the others' added, in forward and
input-gradient passes of the pair-stationary fp16 kernels, on either side of the rule; and the identity map written, not added."""
import numpy as np
import pytest
import torch

from tests.test_gpu_fp32_parts import exact

pytestmark = pytest.mark.gpu


def thin_map(n, full, k_vol=27):
    """Random eighths of the rows through every offset; through offset `full` (None: no such) all of them, in no order."""
    rng = np.random.default_rng(n)
    ins, outs = [], []
    for k in range(k_vol):
        m = n if k == full else n // 8 + k
        outs.append(np.sort(rng.permutation(n)[:m]))
        ins.append(rng.permutation(n)[:m])
    kpos = np.concatenate([[0], np.cumsum([len(o) for o in outs])])
    return tuple(torch.from_numpy(t.astype(np.int32)).cuda() for t in (kpos, np.concatenate(ins), np.concatenate(outs)))


@pytest.mark.parametrize("n,c_in,c_out,full,launches", [(33001, 256, 256, 13, 2), (33001, 256, 256, None, 1), (20000, 256, 256, 13, 1),
                                                        (52001, 128, 128, 0, 2), (30000, 128, 128, 26, 1), (52001, 96, 128, 26, 2)])
def test_whole_numbers(n, c_in, c_out, full, launches):
    """Small whole numbers: every sum is exact, so a row written twice, added twice or left out shows."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    maps = thin_map(n, full)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half() - (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half()
    x, w, g = few(n, c_in), few(27, c_in, c_out), few(n, c_out)
    want = exact(x.float(), w.float(), g.float(), maps[0].tolist(), maps[1].long(), maps[2].long())
    assert max(t.abs().max() for t in want[:2]) < 2048
    plan = capi.Plan(*maps, n, n)
    view, swapped = plan.transposed(), (maps[0], maps[2], maps[1])

    def launched(call):
        capi.profile_reset()
        capi.profile_enable(True)
        call()
        torch.cuda.synchronize()
        capi.profile_enable(False)
        return [q[0] for q in capi.profile_records() if q[0].startswith(("gms_wide", "gms_pairs", "gms_rows"))]

    for p, m, a, b in ((plan, maps, x, g), (view, swapped, None, None)):
        if a is None:                                     # (the transposed plan: the same map the other way round)
            up = exact(g.float(), w.transpose(1, 2).float(), x.float(), m[0].tolist(), m[1].long(), m[2].long())[0]
            out = torch.full_like(x, float("nan"))
            names = launched(lambda: capi.conv_fwd(g, w.transpose(1, 2).contiguous(), out, *m, plan=p))
            assert torch.equal(out.double(), up), names
            continue
        out, gin = torch.full_like(g, float("nan")), torch.full_like(x, float("nan"))
        names = launched(lambda: capi.conv_fwd(a, w, out, *m, plan=p))
        assert len(names) == launches and all(q.startswith("gms_wide" if c_out == 256 else "gms_pairs") for q in names), names
        assert torch.equal(out.double(), want[0])
        names = launched(lambda: capi.conv_bwd(b, a, w, gin, None, *m, plan=p))
        assert torch.equal(gin.double(), want[1]), names
        # added to what is there: no first launch
        again = out.clone()
        assert len(launched(lambda: capi.fusion_fwd(a, w, 0, again, m[0], None, m[1], m[2], False, False, plan=p))) == 1
        assert torch.equal(again.double(), 2 * want[0])
    view.close()
    plan.close()


@pytest.mark.parametrize("how", ["shuffled", "fewer", "more", "none"])
@pytest.mark.parametrize("c_in,c_out", [(256, 256), (128, 128), (256, 128), (128, 256)])
def test_lists_rewritten_under_the_plan(c_in, c_out, how):
    """The offset that met every row, in order, when the plan was made, meets others since (in any order, not all of them, some of them
    twice, or none), and the other offsets have its pairs: the sums are those of the lists as they are."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    n, full = 52001, 13
    rng = np.random.default_rng(c_in + c_out)
    sizes = [n if k == full else n // 8 + k for k in range(27)]
    ins, outs = ([np.arange(n) if k == full else pick(rng.permutation(n)[:m]) for k, m in enumerate(sizes)] for pick in (lambda r: r, np.sort))
    lists = lambda parts: torch.from_numpy(np.concatenate(parts).astype(np.int32)).cuda()
    starts = lambda parts: torch.from_numpy(np.cumsum([0] + [len(p) for p in parts]).astype(np.int32)).cuda()
    maps = starts(outs), lists(ins), lists(outs)
    plan = capi.Plan(*maps, n, n)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half() - (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half()
    x, w, g = few(n, c_in), few(27, c_in, c_out), few(n, c_out)

    def check(beyond=False):
        m = tuple(t.long() for t in maps[1:])
        kpos = maps[0].tolist()
        want = exact(x.float(), w.float(), g.float(), kpos, *m)
        hit = [torch.zeros(n, dtype=torch.bool, device="cuda") for _ in range(2)]
        if beyond:
            w[full, 3, 5], w[full, 2, 1] = float("inf"), float("nan")
            for h, q in zip(hit, (m[1], m[0])):
                h[q[kpos[full]:kpos[full + 1]]] = True
        out, gin = torch.full_like(g, float("nan")), torch.full_like(x, float("nan"))
        capi.conv_fwd(x, w, out, *maps, plan=plan)
        capi.conv_bwd(g, x, w, gin, None, *maps, plan=plan)
        for got, ref, h in ((out, want[0], hit[0]), (gin, want[1], hit[1])):
            assert torch.equal(got[~h].double(), ref[~h])

    check()
    changed = {"shuffled": n, "fewer": n - 777, "more": n + 555, "none": 0}[how]
    rows = [rng.permutation(n) for _ in range(2)]
    rows = [np.concatenate([r, r[:555]])[:changed] for r in rows]
    extra = sizes[full] - changed
    ins[full], outs[full] = rows
    if extra < 0:
        ins[0], outs[0] = ins[0][:extra], outs[0][:extra]
    else:
        ins[20], outs[20] = (np.concatenate([q[20], rng.permutation(n)[:extra]]) for q in (ins, outs))
    for t, new in zip(maps, (starts(outs), lists(ins), lists(outs))):
        t.copy_(new)
    check()
    check(beyond=True)
    plan.close()


@pytest.mark.parametrize("c_in,c_out", [(256, 256), (256, 128)])
@pytest.mark.parametrize("other", [(55000, 27), (52001, 32)], ids=["rows", "offsets"])
def test_plan_of_another_map(other, c_in, c_out):
    """Rows or offsets that do not fit the call's: what that plan says about an offset is not taken over."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    n = 52001
    maps, others = thin_map(n, None), thin_map(other[0], other[1] - 1, other[1])
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    few = lambda *s: (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half() - (torch.randint(0, 64, s, generator=gen, device="cuda") < 3).half()
    x, w, g = few(n, c_in), few(27, c_in, c_out), few(n, c_out)
    want = exact(x.float(), w.float(), g.float(), maps[0].tolist(), maps[1].long(), maps[2].long())
    plan = capi.Plan(*others, other[0], other[0])
    out, gin = torch.full_like(g, float("nan")), torch.full_like(x, float("nan"))
    capi.conv_fwd(x, w, out, *maps, plan=plan)
    capi.conv_bwd(g, x, w, gin, None, *maps, plan=plan)
    assert torch.equal(out.double(), want[0]) and torch.equal(gin.double(), want[1])
    plan.close()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("c_in,c_out", [(64, 64), (128, 256), (32, 96)])
def test_identity_map_added_and_written(c_in, c_out, dtype):
    """The centre offset kept apart on a map without a plan: written by the one entry, added by the other."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    n, k_vol = 2311, 27
    maps = thin_map(n, None)
    kpos = maps[0].tolist()
    keep = torch.cat([torch.arange(kpos[0], kpos[13]), torch.arange(kpos[14], kpos[27])]).cuda()
    cut = maps[0].clone()
    cut[14:] -= kpos[14] - kpos[13]
    imap, omap = maps[1][keep].contiguous(), maps[2][keep].contiguous()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(c_in)
    draw = lambda *s: torch.randint(-1, 2, s, generator=gen, device="cuda").to(dtype)
    x, w = draw(n, c_in), draw(k_vol, c_in, c_out)
    rows = torch.arange(n, dtype=torch.int32, device="cuda")
    whole = [torch.cat([t[:kpos[13]], rows, t[kpos[13]:]]) for t in (imap, omap)]
    full = maps[0].clone()
    full[14:] = cut[14:] + n
    want = exact(x.float(), w.float(), torch.zeros(n, c_out, device="cuda"), full.tolist(), whole[0].long(), whole[1].long())[0]
    out = torch.zeros(n, c_out, dtype=dtype, device="cuda")
    capi.fusion_fwd(x, w, 0, out, cut, None, imap, omap, True, False)
    assert want.abs().max() < 2048 and torch.equal(out.double(), want)
    base = draw(n, c_out)
    out = base.clone()
    knnz = (cut[1:] - cut[:-1]).cpu()
    capi.seq_fwd(x, w, imap.numel(), out, knnz, cut, imap, omap, True, False)
    assert torch.equal(out.double(), want + base.double())
