"""Performance cases of the sparse-convolution path: what a user's program has it do, through the
public entry points (``FGMS.nn`` and ``FGMS.backend``), from a single small object to a merged
LiDAR sweep.

A case is a dict of plain values:

``task``     what the program does in one pass
    ``infer``   one layer, forward, weights under ``fgms_weights_pin`` where ``pinned``
    ``train``   one layer, forward and backward (``FGMS.nn.sparse_conv`` under autograd)
    ``stem``    the same for a network's first layer: its input features need no gradient
    ``updown``  a stride-2 layer and the transposed layer over the same map, forward and backward
    ``scene``   a new point cloud: kernel maps from coordinates at two resolutions, then five
                layers over them, forward and backward
    ``dropin``  the reference's calls on caller-owned buffers, centre offset kept apart
                (``separate_mid``): ``fgms_fusion_fwd_cuda`` and ``fgms_bwd_cuda``
``cloud``    ``indoor`` (sheets and small boxes), ``lidar`` (rings of a spinning sensor, walls),
             ``scattered`` (a random quarter of an indoor cloud)
``order``    row order of the voxels: ``sorted`` by coordinate, or ``scan``, as acquired
``voxels``   input voxels
``kernel``   3 or 5 (submanifold), 2 (stride 2)
``c_in``, ``c_out``, ``dtype`` (``fp16``, ``fp32``, ``tf32``: fp32 tensors with ``allow_tf32``)
"""
import math

import torch

from FGMS import backend
from FGMS.nn import KernelMap, sparse_conv
from fgms_amd import capi, clouds
from fgms_amd.harness import kpos_quantized

# input pairs per output voxel of a 3x3x3 / 5x5x5 submanifold map on these clouds, measured; for work()
_PAIRS = {("indoor", 3): 10.5, ("lidar", 3): 9.8, ("scattered", 3): 3.3,
          ("indoor", 5): 29.0, ("lidar", 5): 26.0, ("scattered", 5): 7.8}


def _case(task, cloud, order, voxels, kernel, c_in, c_out, dtype, pinned=False):
    return dict(task=task, cloud=cloud, order=order, voxels=voxels, kernel=kernel, c_in=c_in, c_out=c_out,
                dtype=dtype, pinned=pinned)


def listed():
    named = [
        # a single object, or the deepest level of a small network: launches and host work
        ("object-2k-32x32-fp16-infer", _case("infer", "indoor", "sorted", 2000, 3, 32, 32, "fp16")),
        # a small room in full precision: the benchmark's plumbing configuration
        ("room-20k-32x32-fp32-train", _case("train", "indoor", "sorted", 20000, 3, 32, 32, "fp32")),
        # a colour stem with a wide kernel: three input channels, 125 offsets
        ("stem-77777-k5-3x32-fp16-train", _case("stem", "indoor", "scan", 77777, 5, 3, 32, "fp16")),
        # the usual first layer: position and intensity, memory-bound
        ("stem-200k-4x32-fp16-train", _case("stem", "indoor", "sorted", 200000, 3, 4, 32, "fp16")),
        # the ordinary layer of an indoor network, mixed precision (the headline workload)
        ("indoor-200k-64x64-fp16-train", _case("train", "indoor", "sorted", 200000, 3, 64, 64, "fp16")),
        # the same in fp32 with products allowed in tf32
        ("indoor-200k-64x64-tf32-train", _case("train", "indoor", "sorted", 200000, 3, 64, 64, "tf32")),
        # merged LiDAR sweeps, wide layer, rows as the sensor delivered them
        ("lidar-120k-128x128-fp16-train", _case("train", "lidar", "scan", 120000, 3, 128, 128, "fp16")),
        # one resolution step down and up again, sharing a map
        ("updown-200k-64x128-fp16-train", _case("updown", "indoor", "sorted", 200000, 2, 64, 128, "fp16")),
        # wide layer over a thinned cloud, inference with constant weights
        ("scattered-50k-256x256-fp16-infer", _case("infer", "scattered", "sorted", 50000, 3, 256, 256, "fp16", True)),
        # an output layer: the number of classes is no multiple of anything
        ("head-60001-96x20-fp16-train", _case("train", "indoor", "sorted", 60001, 3, 96, 20, "fp16")),
        # a program written for the reference, channel counts off the powers of two
        ("dropin-90k-48x96-fp16", _case("dropin", "lidar", "sorted", 90000, 3, 48, 96, "fp16")),
        # a data loader hands over a new sweep every iteration: maps and plans are built each time
        ("scene-100k-32-fp16-train", _case("scene", "lidar", "scan", 100000, 3, 32, 32, "fp16")),
    ]
    return [dict(c, name=n) for n, c in named]


# channel counts in use at each kind of layer (the shape sweep of the tests walks the same ones)
_NARROW, _MIDDLE, _WIDE = (3, 4, 5, 6, 8), (16, 24, 32, 48, 64, 96), (96, 128, 160, 256)


def draw(rng):
    task = rng.choice(("infer", "infer", "train", "train", "train", "stem", "updown", "scene", "dropin", "head", "wide", "wide"))
    cloud = rng.choice(("indoor", "indoor", "lidar"))
    order = rng.choice(("sorted", "sorted", "scan"))
    dtype = rng.choice(("fp16", "fp16", "fp16", "fp32", "tf32"))

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if task == "stem":
        k = rng.choice((3, 3, 5))
        return _case("stem", cloud, order, size(5000, 200000 if k == 3 else 80000), k, rng.choice(_NARROW), rng.choice((16, 32, 64) if k == 3 else (16, 32)), dtype)
    if task == "updown":
        c = rng.choice((32, 48, 64, 96))
        return _case("updown", cloud, order, size(5000, 200000), 2, c, rng.choice((c, 2 * c) if c < 96 else (c, 128)), dtype)
    if task == "scene":
        return _case("scene", cloud, order, size(5000, 100000), 3, rng.choice((16, 32)), 32, rng.choice(("fp16", "fp16", "fp32")))
    if task == "head":
        return _case("train", cloud, order, size(5000, 60000), 3, rng.choice((32, 64, 96)), rng.randrange(13, 29), rng.choice(("fp16", "fp32")))
    if task == "wide":
        c = rng.choice(_WIDE)
        most = 40000 if c > 128 else 100000
        if rng.random() < 0.5:
            return _case("infer", "scattered", order, size(2000, 50000), 3, c, rng.choice((128, 256)), dtype, rng.random() < 0.5)
        return _case("train", cloud, order, size(2000, most), 3, c, c if c <= 160 else 128, "fp16" if most * c * c > 1 << 30 else dtype)
    if task == "dropin":
        return _case("dropin", cloud, order, size(2000, 100000), 3, rng.choice(_MIDDLE), rng.choice(_MIDDLE), rng.choice(("fp16", "fp16", "fp32")))
    return _case(task, cloud, order, size(1000, 200000), 3, rng.choice(_MIDDLE[:5]), rng.choice(_MIDDLE[:5]), dtype,
                 task == "infer" and rng.random() < 0.5)


# ------------------------------------------------------------------------------- point clouds
def _indoor_points(n, gen):
    """Points of planar patches (every second one oblique) and of small ones (furniture), half a
    voxel apart, in a room whose size grows with the cloud."""
    scale = min(1.0, math.sqrt(n / 50000.0))
    patches = max(8, int(1.5 * n / (5600.0 * scale * scale)))
    room = 512.0 * (max(n, 2000) / 200000.0) ** (1.0 / 3.0)
    dev = gen.device

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=gen, device=dev)

    small = (torch.arange(patches, device=dev) % 3 == 2).float().view(-1, 1)
    half = (uniform(22, 42, patches, 2) * (1 - small) + uniform(8, 18, patches, 2) * small) * scale
    centre = uniform(0.15 * room, 0.85 * room, patches, 3)
    normal = torch.randn(patches, 3, generator=gen, device=dev)
    axis = torch.nn.functional.one_hot(torch.randint(0, 3, (patches,), generator=gen, device=dev), 3).float()
    oblique = (torch.arange(patches, device=dev) % 2 == 1).view(-1, 1)
    normal = torch.where(oblique, normal / normal.norm(dim=1, keepdim=True), axis)
    other = torch.nn.functional.one_hot(normal.abs().argmin(1), 3).float()
    u = torch.linalg.cross(normal, other)
    u = u / u.norm(dim=1, keepdim=True)
    v = torch.linalg.cross(normal, u)
    r = int(math.ceil(42 * scale)) * 2
    step = torch.arange(-r, r + 1, device=dev).float() * 0.5
    a, b = torch.meshgrid(step, step, indexing="ij")
    a, b = a.reshape(1, -1), b.reshape(1, -1)
    pts = centre[:, None] + a[..., None] * u[:, None] + b[..., None] * v[:, None]
    keep = (a.abs() <= half[:, :1]) & (b.abs() <= half[:, 1:])
    return pts[keep]


def _lidar_points(n, gen):
    """Hits of a 64-beam sensor, 1.73 m over the ground among box obstacles, from positions along
    its way, in voxels of 5 cm."""
    dev = gen.device
    azimuths = max(128, min(2048, int(2048 * n / 90000.0)))
    sweeps = 6 if n <= 120000 else 12
    elev = torch.deg2rad(torch.linspace(-25.0, 3.0, 64, device=dev))
    azim = torch.arange(azimuths, device=dev) * (2 * math.pi / azimuths)
    aa, ee = torch.meshgrid(azim, elev, indexing="ij")
    d = torch.stack([torch.cos(ee) * torch.cos(aa), torch.cos(ee) * torch.sin(aa), torch.sin(ee)], -1).reshape(-1, 3)

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=gen, device=dev)

    ang, rad = uniform(0, 2 * math.pi, 60), uniform(5, 45, 60)
    half = torch.stack([uniform(0.8, 5, 60), uniform(0.8, 5, 60), uniform(0.7, 4, 60)], 1)
    centre = torch.stack([rad * torch.cos(ang), rad * torch.sin(ang), half[:, 2]], 1)
    pts = []
    for s in range(sweeps):
        origin = torch.tensor([2.3 * s, 0.6 * s, 1.73], device=dev)
        t = torch.where(d[:, 2] < -1e-6, -origin[2] / d[:, 2], torch.full_like(d[:, 2], math.inf))
        inv = 1.0 / torch.where(d.abs() < 1e-7, torch.full_like(d, 1e-7), d)
        for c, h in zip(centre, half):
            t0, t1 = (c - h - origin) * inv, (c + h - origin) * inv
            near, far = torch.minimum(t0, t1).amax(1), torch.maximum(t0, t1).amin(1)
            t = torch.where((near <= far) & (near > 0) & (near < t), near, t)
        ok = (t >= 2.0) & (t <= 50.0)
        t = t + 0.01 * torch.randn(t.shape, generator=gen, device=dev)
        pts.append((origin + d * t[:, None])[ok])
    return torch.cat(pts) / 0.05


def _voxels(case, gen):
    """int32 [voxels, 3]: exactly as many as the case says, a slab of the cloud along x."""
    n = case["voxels"]
    want = 4 * n if case["cloud"] == "scattered" else n
    make = _lidar_points if case["cloud"] == "lidar" else _indoor_points
    pts = make(want, gen)
    while True:
        v = torch.floor(pts).long()
        v = v - v.amin(0)
        key = (v[:, 0] << 40) | (v[:, 1] << 20) | v[:, 2]
        uniq, inverse = torch.unique(key, return_inverse=True)
        if uniq.numel() >= want:
            break
        pts = torch.cat([pts, make(want, gen) + (pts.amax(0) + 8) * torch.tensor([1.0, 0, 0], device=pts.device)])
    first = torch.full((uniq.numel(),), key.numel(), device=key.device).scatter_reduce_(
        0, inverse, torch.arange(key.numel(), device=key.device), "amin")
    rows = torch.arange(want, device=key.device)
    if case["cloud"] == "scattered":
        rows = torch.randperm(want, generator=gen, device=key.device)[:n].sort().values
    if case["order"] == "scan":
        rows = rows[first[rows].argsort()]
    k = uniq[rows]
    return torch.stack([k >> 40, (k >> 20) & 0xFFFFF, k & 0xFFFFF], 1).int().contiguous()


def _coarse(vox):
    """The stride-2 output voxels, as the data loader hands them over."""
    return torch.unique(torch.div(vox, 2, rounding_mode="floor"), dim=0).int().contiguous()


# ------------------------------------------------------------------------------- one pass
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dt = torch.float16 if case["dtype"] == "fp16" else torch.float32
    task, ci, co = case["task"], case["c_in"], case["c_out"]
    vox = _voxels(case, gen)
    n = vox.shape[0]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda").to(dt)

    def weight(k_vol, a, b):
        bound = 1.0 / math.sqrt(k_vol * a)
        return ((torch.rand(k_vol, a, b, generator=gen, device="cuda") * 2 - 1) * bound).to(dt)

    s = {"task": task, "tf32": case["dtype"] == "tf32"}
    if task == "scene":
        c = case["c_in"]
        s.update(vox=vox, coarse=_coarse(vox), offs3=clouds.offsets_cube(3), offs2=clouds.offsets_cube(2),
                 x=torch.rand(n, 4, generator=gen, device="cuda").to(dt), g=normal(n, case["c_out"]),
                 w=[weight(27, 4, c), weight(27, c, c), weight(8, c, 2 * c), weight(27, 2 * c, 2 * c), weight(8, 2 * c, case["c_out"])])
        for w in s["w"]:
            w.requires_grad_()
        return s
    offsets = clouds.offsets_cube(case["kernel"])
    if task == "updown":
        s.update(kmap=KernelMap.from_coords(vox, _coarse(vox), offsets, stride=2), x=normal(n, ci).requires_grad_(),
                 w1=weight(8, ci, co).requires_grad_(), w2=weight(8, co, ci).requires_grad_(), g=normal(n, ci))
        s["up"] = s["kmap"].transposed()
        return s
    k_vol = len(offsets)
    w = weight(k_vol, ci, co)
    if task == "dropin":
        imap, omap, knnz, kpos = capi.build_kernel_map(vox, vox, offsets, skip_offset=k_vol // 2)
        knnz = knnz.cpu()
        qkpos, qsum = kpos_quantized(knnz, kpos, k_vol, 256)
        s.update(imap=imap.clone(), omap=omap.clone(), kpos=kpos, qkpos=qkpos, qsum=qsum, x=normal(n, ci), w=w, g=normal(n, co))
        return s
    x = torch.rand(n, ci, generator=gen, device="cuda").to(dt) if task == "stem" else normal(n, ci)
    s.update(kmap=KernelMap.from_coords(vox, vox, offsets), x=x, w=w)
    if task == "infer":
        if case["pinned"]:
            backend.fgms_weights_pin(w)
    else:
        s.update(g=normal(n, co))
        w.requires_grad_()
        if task == "train":
            x.requires_grad_()
    return s


def run(s):
    task, tf32 = s["task"], s["tf32"]
    if task == "infer":
        with torch.no_grad():
            return sparse_conv(s["x"], s["w"], s["kmap"], tf32)
    if task in ("train", "stem"):
        y = sparse_conv(s["x"], s["w"], s["kmap"], tf32)
        inputs = (s["x"], s["w"]) if task == "train" else (s["w"],)
        return (y.detach(),) + torch.autograd.grad(y, inputs, s["g"])
    if task == "updown":
        y = sparse_conv(sparse_conv(s["x"], s["w1"], s["kmap"], tf32), s["w2"], s["up"], tf32)
        return (y.detach(),) + torch.autograd.grad(y, (s["x"], s["w1"], s["w2"]), s["g"])
    if task == "scene":
        fine = KernelMap.from_coords(s["vox"], s["vox"], s["offs3"])
        down = KernelMap.from_coords(s["vox"], s["coarse"], s["offs2"], stride=2)
        low = KernelMap.from_coords(s["coarse"], s["coarse"], s["offs3"])
        w = s["w"]
        y = sparse_conv(sparse_conv(s["x"], w[0], fine, tf32), w[1], fine, tf32)
        y = sparse_conv(sparse_conv(y, w[2], down, tf32), w[3], low, tf32)
        y = sparse_conv(y, w[4], down.transposed(), tf32)
        return (y.detach(),) + torch.autograd.grad(y, w, s["g"])
    x, w, g = s["x"], s["w"], s["g"]
    maps = (s["kpos"], s["qkpos"], s["imap"], s["omap"])
    out = torch.zeros(x.shape[0], w.shape[2], dtype=x.dtype, device=x.device)
    backend.fgms_fusion_fwd_cuda(x, w, s["qsum"], out, *maps, True, tf32)
    gx, gw = torch.zeros_like(x), torch.zeros_like(w)
    backend.fgms_bwd_cuda(g, x, w, s["qsum"], gx, gw, *maps, True, tf32)
    return out, gx, gw


# ------------------------------------------------------------------------------- what it takes
def work(case):
    """Every input (features, weights, output gradient, pair lists or coordinates) read once, every
    output written once; two operations per pair, channel and channel, for each product."""
    esz = 2 if case["dtype"] == "fp16" else 4
    n, ci, co, task = case["voxels"], case["c_in"], case["c_out"], case["task"]
    if task == "scene":
        pairs = _PAIRS[case["cloud"], 3]
        low = 0.31 * n                      # coarse voxels
        layers = [(pairs * n, 4, ci, 2), (pairs * n, ci, ci, 3), (n, ci, 2 * ci, 3), (pairs * low, 2 * ci, 2 * ci, 3), (n, 2 * ci, co, 3)]
        weights = 27 * (4 * ci + ci * ci + 4 * ci * ci) + 8 * 2 * ci * (ci + co)
        return {"bytes": 12 * (n + low) + esz * (n * (4 + 2 * co) + 2 * weights),
                "flops": sum(2.0 * m * a * b * passes for m, a, b, passes in layers)}
    if task == "updown":
        return {"bytes": 8 * n + esz * (n * ci * 4 + 2 * 2 * 8 * ci * co), "flops": 2 * 3 * 2.0 * n * ci * co}
    pairs = _PAIRS[case["cloud"], case["kernel"]] * n
    weights = case["kernel"] ** 3 * ci * co
    passes = {"infer": 1, "stem": 2}.get(task, 3)
    bytes_ = {"infer": n * (ci + co) + weights, "stem": n * (ci + 2 * co) + 2 * weights}.get(task, n * 2 * (ci + co) + 2 * weights)
    return {"bytes": 8 * pairs + esz * bytes_, "flops": 2.0 * pairs * ci * co * passes}


def tolerance(case):
    """fp16 results are rounded once (2^-11 of the value), some of them sums of a few rounded parts;
    tf32 mode keeps at least the 2^-11 of its products' inputs, and its sums are fp32."""
    if case["dtype"] == "fp16":
        return {"rel": 2e-3}
    return {"rel": 1e-4 if case["dtype"] == "tf32" else 1e-5}
