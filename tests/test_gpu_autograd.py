"""FGMS.nn: the autograd Function / Module over FGMS.backend, against torch's own autograd
through the index_add formulation of the same convolution (float64 on the GPU)."""
import numpy as np
import pytest
import torch

from fgms_amd import clouds
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def reference(x, w, kmap):
    out = torch.zeros(kmap.n_out, w.shape[2], dtype=torch.float64, device=x.device)
    kpos = kmap.kpos.cpu().tolist()
    for k in range(kmap.k_vol):
        i, o = kmap.in_map[kpos[k]:kpos[k + 1]].long(), kmap.out_map[kpos[k]:kpos[k + 1]].long()
        out.index_add_(0, o, x[i] @ w[k])
    return out


def small_layer(seed, c_in, c_out, dtype, strided=False):
    rng = np.random.default_rng(seed)
    pts = np.concatenate([clouds._patch(rng, rng.uniform(6, 18, 3), 9, 9, oblique=False),
                          clouds._sphere_shell(rng, np.array([12., 12, 12]), 7.0, 2500)])
    vox = clouds.dedup(pts, 24)
    if not strided:
        return clouds.submanifold_case(vox, c_in, c_out, dtype, rng)
    coarse = clouds.downsample_coords(vox, 2)
    imap, omap, knnz, kpos = clouds.build_kernel_map(vox, coarse, clouds.offsets_cube(2), 2)
    return clouds.make_layer(rng, imap, omap, knnz, kpos, len(vox), len(coarse), c_in, c_out, dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("strided", [False, True], ids=["submanifold", "stride2"])
def test_function_matches_torch_autograd(dtype, strided):
    from FGMS import nn as fnn
    L = small_layer(41, 64, 32, dtype, strided)
    D = G.to_dev(L)
    kmap = fnn.KernelMap(D["imap"], D["omap"], L["knnz"], L["n_in"], L["n_out"])
    x = D["in_feats"].clone().requires_grad_(True)
    w = D["kernel"].clone().requires_grad_(True)
    y = fnn.sparse_conv(x, w, kmap)
    (y.float() * D["out_grad"].float()).sum().backward()

    x64 = D["in_feats"].double().requires_grad_(True)
    w64 = D["kernel"].double().requires_grad_(True)
    y64 = reference(x64, w64, kmap)
    (y64 * D["out_grad"].double()).sum().backward()
    mode = G.mode_of(dtype)
    G.assert_close(y.detach().cpu().numpy(), y64.detach().cpu().numpy(), mode, "forward")
    G.assert_close(x.grad.cpu().numpy(), x64.grad.cpu().numpy(), mode, "grad feats")
    G.assert_close(w.grad.cpu().numpy(), w64.grad.cpu().numpy(), mode, "grad weight")

    # the transposed map runs the same pairs backwards: its forward is the input gradient
    yt = fnn.sparse_conv(D["out_grad"], w.detach().transpose(1, 2).contiguous(), kmap.transposed())
    G.assert_close(yt.cpu().numpy(), x64.grad.cpu().numpy(), mode, "transposed forward")


def test_module_trains():
    from FGMS import nn as fnn
    torch.manual_seed(0)
    L = small_layer(42, 16, 32, np.float32)
    D = G.to_dev(L)
    kmap = fnn.KernelMap(D["imap"], D["omap"], L["knnz"], L["n_in"], L["n_out"])
    l1 = fnn.SparseConv(16, 32, 27, bias=True, device="cuda")
    l2 = fnn.SparseConv(32, 8, 27, device="cuda")
    target = torch.randn(L["n_out"], 8, device="cuda")
    opt = torch.optim.SGD(list(l1.parameters()) + list(l2.parameters()), lr=0.05)
    losses = []
    for _ in range(8):
        opt.zero_grad()
        y = l2(torch.relu(l1(D["in_feats"], kmap)), kmap)     # both layers share the map and its plan
        loss = ((y - target) ** 2).mean()
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    assert losses[-1] < losses[0] and all(np.isfinite(losses))
    from FGMS import backend
    assert backend.fgms_plan_cache_size() >= 1


def test_kernel_map_from_coordinates():
    from FGMS import nn as fnn
    rng = np.random.default_rng(43)
    vox = clouds.dedup(clouds._sphere_shell(rng, np.array([12., 12, 12]), 7.0, 2500), 24)
    want = clouds.build_kernel_map(vox, vox, clouds.offsets_cube(3))
    kmap = fnn.KernelMap.from_coords(torch.from_numpy(vox).cuda(), torch.from_numpy(vox).cuda(),
                                     clouds.offsets_cube(3))
    assert np.array_equal(kmap.in_map.cpu().numpy(), want[0])
    assert np.array_equal(kmap.out_map.cpu().numpy(), want[1])
    assert np.array_equal(kmap.kernel_nnz.numpy(), want[2])
    y = fnn.sparse_conv(torch.randn(len(vox), 32, device="cuda"), torch.randn(27, 32, 32, device="cuda"), kmap)
    assert y.shape == (len(vox), 32) and torch.isfinite(y).all()


def test_kernel_map_checks_its_sizes():
    from FGMS import nn as fnn
    e = torch.zeros(5, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        fnn.KernelMap(e, e, [2, 2], 10, 10)          # 4 != 5 pairs
    kmap = fnn.KernelMap(e, e, [2, 3], 10, 10)
    with pytest.raises(ValueError):
        fnn.sparse_conv(torch.zeros(9, 4, device="cuda"), torch.zeros(2, 4, 4, device="cuda"), kmap)


@pytest.fixture
def one_layer():
    from FGMS import nn as fnn
    L = small_layer(44, 32, 48, np.float32)
    D = G.to_dev(L)
    kmap = fnn.KernelMap(D["imap"], D["omap"], L["knnz"], L["n_in"], L["n_out"])
    return D["in_feats"], D["kernel"], D["out_grad"], kmap


def test_tangents_are_refused(one_layer):
    """No forward-mode derivative exists: an input with a tangent must not come out as one without."""
    import torch.autograd.forward_ad as fwd
    from FGMS import nn as fnn
    x, w, g, kmap = one_layer
    with fwd.dual_level():
        for feats, weight in ((fwd.make_dual(x, x), w), (x, fwd.make_dual(w, w))):
            with pytest.raises(NotImplementedError, match="tangent"):
                fnn.sparse_conv(feats, weight, kmap)
        leaf = x.clone().requires_grad_(True)
        y = fnn.sparse_conv(leaf, w, kmap)
        with pytest.raises(NotImplementedError, match="tangent"):
            torch.autograd.grad(y, leaf, fwd.make_dual(g, g))
        assert fwd.unpack_dual(fnn.sparse_conv(x, w, kmap)).tangent is None
    for transform in (torch.func.vmap, lambda f: torch.func.grad(lambda t: f(t).sum()), lambda f: lambda t: torch.func.jvp(f, (t,), (t,))):
        with pytest.raises(RuntimeError):
            transform(lambda t: fnn.sparse_conv(t, w, kmap))(x[None] if transform is torch.func.vmap else x)


def test_saved_tensor_hooks(one_layer):
    """Offloading hooks and checkpointing give the plain gradients; a hook that hands back something other
    than what was saved is an error, not a read past its end."""
    from torch.utils.checkpoint import checkpoint
    from FGMS import nn as fnn
    x0, w0, g, kmap = one_layer

    def grads(layer, unpack=None, offload=False):
        x, w = x0.clone().requires_grad_(True), w0.clone().requires_grad_(True)
        if offload:
            with torch.autograd.graph.save_on_cpu():
                y = layer(x, w)
        elif unpack:
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
                y = layer(x, w)
        else:
            y = layer(x, w)
        return torch.autograd.grad(y, (x, w), g)

    conv = lambda x, w: fnn.sparse_conv(x, w, kmap)
    want = grads(conv)
    strided = lambda t: t.detach().transpose(0, 1).contiguous().transpose(0, 1)
    for got in (grads(conv, offload=True), grads(conv, unpack=strided),
                grads(lambda x, w: checkpoint(conv, x, w, use_reentrant=False))):
        for a, b in zip(got, want):          # (sums of atomics: equal up to their order)
            G.assert_close(a.cpu().numpy(), b.cpu().numpy(), "fp32")
    for wrong in (lambda t: t.detach().half(), lambda t: t.detach().cpu(), lambda t: t.detach()[:-1], lambda t: t.detach()[..., :4],
                  lambda t: t.detach().reshape(-1)):
        with pytest.raises(ValueError, match="came back"):
            grads(conv, unpack=wrong)


def test_traced_layer_is_recorded(one_layer, tmp_path):
    """torch.jit.trace records the call, not its result: other inputs give other outputs, gradients included."""
    from FGMS import nn as fnn
    x, w, g, kmap = one_layer

    class Net(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.conv = fnn.SparseConv(w.shape[1], w.shape[2], 27, device="cuda")

        def forward(self, t):
            return torch.relu(self.conv(t, kmap))

    net = Net()
    traced = torch.jit.trace(net, x, check_trace=False)
    torch.jit.save(traced, str(tmp_path / "net.pt"))
    other = torch.randn_like(x)
    with torch.no_grad():
        net.conv.weight.mul_(-0.5)             # (the trace shares the module's parameter)
    for run, scale in ((traced, 1.0), (torch.jit.load(str(tmp_path / "net.pt")), -2.0)):
        a, b = other.clone().requires_grad_(True), other.clone().requires_grad_(True)
        y = run(a)
        z = torch.relu(fnn.sparse_conv(b, net.conv.weight.detach() * scale, kmap))
        G.assert_close(y.detach().cpu().numpy(), z.detach().cpu().numpy(), "fp32")
        G.assert_close(torch.autograd.grad(y, a, g)[0].cpu().numpy(), torch.autograd.grad(z, b, g)[0].cpu().numpy(), "fp32")


def test_threads_drop_each_others_plans():
    """Forward and backward passes of several threads over more maps than the plan cache holds."""
    import threading
    from FGMS import backend, nn as fnn
    backend.fgms_plan_cache(True, 1)
    failures = []

    def work(seed):
        try:
            L = small_layer(seed, 32, 32, np.float16)
            with torch.cuda.stream(torch.cuda.Stream()):
                D = G.to_dev(L)
                kmap = fnn.KernelMap(D["imap"], D["omap"], L["knnz"], L["n_in"], L["n_out"])
                x, w = D["in_feats"].clone().requires_grad_(True), D["kernel"].clone().requires_grad_(True)
                passes = [torch.autograd.grad(fnn.sparse_conv(x, w, kmap), (x, w), D["out_grad"]) for _ in range(25)]
                torch.cuda.current_stream().synchronize()
            for got in passes:
                for a, b in zip(got, passes[0]):
                    G.assert_close(a.cpu().numpy(), b.cpu().numpy(), "fp16")
        except Exception as e:          # noqa: BLE001 (reported by the main thread)
            failures.append(e)

    try:
        threads = [threading.Thread(target=work, args=(60 + i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        backend.fgms_plan_cache(True, 8)
    assert not failures, failures[0]
