"""A captured graph keeps what it points at: later eager calls that need bigger workspaces get new
buffers, the plan cache does not give its plans back, and replays still give the eager results."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def cloud_layer(n_vox, c_in, c_out, dtype):
    rng = np.random.default_rng(n_vox)
    vox = clouds.cloud_indoor(clouds.rng_for(2), target=n_vox)
    return clouds.submanifold_case(vox, c_in, c_out, dtype, rng)


# padded copies on either side and the weight gradient's accumulator; re-laid weights; the generic accumulator
@pytest.mark.parametrize("shape,dtype,policy", [((32, 20), np.float16, 0), ((20, 96), np.float32, 0), ((128, 128), np.float16, 0),
                                                ((20, 12), np.float16, 1)],
                         ids=["fp16 32x20", "fp32 20x96", "fp16 128x128", "fp16 generic"])
def test_replays_after_bigger_calls(shape, dtype, policy):
    from fgms_amd import capi
    capi.set_kernel_policy(policy)
    side = torch.cuda.Stream()
    layers = []
    for n, channels in ((3000, shape), (30000, tuple(2 * c if c % 32 == 0 else c for c in shape))):
        D = G.to_dev(cloud_layer(n, *channels, dtype))
        maps = (D["kpos"], D["imap"], D["omap"])
        outs = [torch.zeros(D["n_out"], channels[1], dtype=D["kernel"].dtype, device="cuda"), torch.zeros_like(D["in_feats"]),
                torch.zeros_like(D["kernel"])]
        layers.append((D, maps, outs, capi.Plan(*maps, D["n_in"], D["n_out"])))

    def run(layer):
        D, maps, outs, plan = layer
        capi.conv_fwd(D["in_feats"], D["kernel"], outs[0], *maps, plan=plan)
        capi.conv_bwd(D["out_grad"], D["in_feats"], D["kernel"], outs[1], outs[2], *maps, plan=plan)
        return outs

    small, big = layers
    side.wait_stream(torch.cuda.current_stream())
    try:
        with torch.cuda.stream(side):
            want = [t.clone() for t in run(small)]
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side, capture_error_mode="thread_local"):
            run(small)
        with torch.cuda.stream(side):
            run(big)                                   # needs bigger workspaces on the same stream
        torch.cuda.synchronize()
        # whatever was given back is in other hands by now
        others = [capi.Plan(*big[1], big[0]["n_in"], big[0]["n_out"]) for _ in range(3)]
        other = torch.cuda.Stream()
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            expect_big = [t.clone() for t in run(big)]
        torch.cuda.synchronize()
        mode = G.mode_of(dtype)
        for _ in range(3):
            for t in small[2]:
                t.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            for got, ref in zip(small[2], want):
                G.assert_close(got.cpu().numpy(), ref.cpu().numpy(), mode, "replay")
            with torch.cuda.stream(side):
                run(big)
            torch.cuda.synchronize()
            for got, ref in zip(big[2], expect_big):
                G.assert_close(got.cpu().numpy(), ref.cpu().numpy(), mode, "eager after a replay")
        for p in others:
            p.close()
    finally:
        capi.set_kernel_policy(0)
        for layer in layers:
            layer[3].close()


def test_replays_after_the_plan_cache_moved_on():
    """A layer recorded through FGMS.nn, then more maps than the cache holds, then an emptied cache."""
    from FGMS import backend, nn as fnn
    backend.fgms_plan_cache(True, 2)
    layers = []
    for n in (2500, 2600, 2700, 2800, 2900):
        L = cloud_layer(n, 64, 64, np.float16)
        D = G.to_dev(L)
        layers.append((D["in_feats"], D["kernel"], fnn.KernelMap(D["imap"], D["omap"], L["knnz"], L["n_in"], L["n_out"])))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    x, w, kmap = layers[0]
    try:
        with torch.cuda.stream(side):
            want = fnn.sparse_conv(x, w, kmap)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = fnn.sparse_conv(x, w, kmap)
        for step in range(3):
            for other in layers[1:]:
                fnn.sparse_conv(*other)
            assert backend.fgms_plan_cache_size() == (3 if step == 0 else 2)   # (the captured map's, and two)
            backend.fgms_plan_cache_clear()
            for other in layers[1:]:                    # (builds that would take the blocks given back)
                fnn.sparse_conv(*other)
            torch.cuda.synchronize()
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            G.assert_close(out.cpu().numpy(), want.cpu().numpy(), "fp16", "replay")
    finally:
        backend.fgms_plan_cache(True, 8)


def test_fp32_capture_in_the_workspace_of_another_mode():
    """A stream that has run a layer in tf32 mode holds 4 bytes a weight: a capture of the layer in fp32 finds a kernel that
    needs no more, and its replays give the eager results."""
    from fgms_amd import capi
    capi.set_kernel_policy(0)
    D = G.to_dev(cloud_layer(9000, 64, 64, np.float32))
    maps = (D["kpos"], D["imap"], D["omap"])
    plan = capi.Plan(*maps, D["n_in"], D["n_out"])
    side, out = torch.cuda.Stream(), torch.empty_like(D["out_grad"])
    want = torch.empty_like(out)
    capi.conv_fwd(D["in_feats"], D["kernel"], want, *maps, plan=plan)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, arch80=True, plan=plan)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side, capture_error_mode="thread_local"):
        capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, plan=plan)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        G.assert_close(out.cpu().numpy(), want.cpu().numpy(), "fp32", "replay")
        with torch.cuda.stream(side):                  # (the buffer grows: the graph keeps the one it points at)
            capi.conv_fwd(D["in_feats"], D["kernel"], out, *maps, plan=plan)
        torch.cuda.synchronize()
        G.assert_close(out.cpu().numpy(), want.cpu().numpy(), "fp32", "eager")
    plan.close()
