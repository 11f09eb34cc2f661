"""The work a user of this framework has it do, as measurable cases.

Every case goes through the public layers (`mappedconvolutions_amd.nn`, `.util`): a training
pass is the forward call plus the gradients autograd returns, an inference pass the forward
call alone.  `listed()` names the cases, `draw()` gives more of the same ranges.
"""
import torch

from mappedconvolutions_amd import nn, util
from mappedconvolutions_amd.util import synthetic

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp64": torch.float64}
SIZE = {"fp32": 4, "bf16": 2, "fp64": 8}


def listed():
    return [
        # One equirectangular image through one 3x3 layer, no gradients: the smallest call, a
        # network's first layer in serving.
        dict(name="conv_small_forward", kind="conv", dtype="fp32", B=1, Ci=16, Co=32, H=64, W=128,
             radius=1, map="latitude", interp="bilinear", train=False, plan=False),
        # An inner layer of a small network in mixed precision, training.
        dict(name="conv_small_train_bf16", kind="conv", dtype="bf16", B=4, Ci=32, Co=64, H=64,
             W=128, radius=1, map="latitude", interp="bilinear", train=True, plan=False),
        # The benchmark's training step: 3x3 on a batch of 256x512 panoramas.
        dict(name="conv_train_fp32", kind="conv", dtype="fp32", B=8, Ci=64, Co=64, H=256, W=512,
             radius=1, map="latitude", interp="bilinear", train=True, plan=False),
        # A real projection map (fractional rows and columns, wrapping at the seam), ragged sizes
        # and channel counts, the layer keeping its map's plan over the epoch.
        dict(name="conv_gnomonic_odd", kind="conv", dtype="fp32", B=3, Ci=24, Co=40, H=125, W=250,
             radius=1, map="gnomonic", interp="bispherical", train=True, plan=True),
        # The largest: an encoder's 5x5 layer on a batch of 512x1024 panoramas in bf16.
        dict(name="conv_encoder_bf16", kind="conv", dtype="bf16", B=16, Ci=128, Co=128, H=512,
             W=1024, radius=2, map="latitude", interp="bilinear", train=True, plan=False),
        # The timing sweep this operator family comes with: float64, few channels, a map of
        # shuffled pixels (no two taps are neighbours).
        dict(name="conv_shuffle_fp64", kind="conv", dtype="fp64", B=1, Ci=10, Co=1, H=200, W=500,
             radius=1, map="shuffle", interp="bilinear", train=True, plan=False),
        # A weighted convolution over the vertices of a level-6 mesh, four vertices per tap.
        dict(name="mesh_train_fp32", kind="mesh", dtype="fp32", B=4, Ci=64, Co=128, V=40962, K=7,
             P=4, map="random", train=True),
        # A decoder's up-sampling layer: the transposed convolution onto twice the resolution.
        dict(name="tconv_decoder_fp32", kind="tconv", dtype="fp32", B=4, Ci=64, Co=32, H=128,
             W=256, factor=2, interp="bilinear", train=True),
        # 3x3 max pooling at full resolution, with the winners and its gradient.
        dict(name="max_pool_train", kind="pool", op="max", dtype="fp32", B=4, C=64, H=512, W=1024,
             stride=1, map="latitude", interp="bilinear"),
        # Average pooling to half the (odd) resolution under a real projection map.
        dict(name="avg_pool_stride2", kind="pool", op="avg", dtype="fp32", B=2, C=32, H=249, W=498,
             stride=2, map="gnomonic", interp="bispherical"),
        # Cube faces onto the equirectangular grid and back: scatter forward, gather backward.
        dict(name="resample_cube", kind="resample", op="resample", dtype="fp32", B=4, C=64, F=256,
             interp="bilinear"),
        # The 8 nearest of a mesh's vertices for every pixel of a panorama.
        dict(name="knn", kind="knn", B=1, D=3, R=40962, Q=524288, k=8),
    ]


def _log(rng, low, high):
    """A whole number between low and high, uniform in its logarithm."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "bf16", "bf16", "fp64", "mesh", "tconv", "max",
                       "avg", "resample", "knn"])
    if kind in ("conv", "bf16"):
        # the dimensions that the cost multiplies are drawn until it is within the largest
        # listed case of the same type
        most = 77e9 if kind == "conv" else 2e12
        while True:
            c = dict(kind="conv", dtype="fp32" if kind == "conv" else "bf16", B=_log(rng, 1, 16),
                     Ci=_log(rng, 3, 128), Co=_log(rng, 8, 128), H=_log(rng, 32, 512),
                     radius=rng.choice([1, 1, 1, 2]))
            c["W"] = 2 * c["H"] + rng.choice([0, 0, 0, 1, 5])
            if 1e7 < _conv_flops(c) / 3 < most:
                break
        c.update(map=rng.choice(["latitude", "gnomonic"]),
                 interp=rng.choice(["bilinear", "bilinear", "bispherical", "nearest"]),
                 train=rng.random() < 0.75, plan=rng.random() < 0.3)
        return c
    if kind == "fp64":
        H = _log(rng, 10, 500)
        return dict(kind="conv", dtype="fp64", B=rng.choice([1, 2]), Ci=_log(rng, 2, 16),
                    Co=_log(rng, 1, 16), H=H, W=_log(rng, H, 2 * H), radius=1, map="shuffle",
                    interp="bilinear", train=rng.random() < 0.75, plan=False)
    if kind == "mesh":
        if rng.random() < 0.5:  # a real mesh kernel: barycentric weights of three vertices
            shape = dict(V=10 * 4 ** rng.choice([3, 4, 5]) + 2, P=3, map="icosphere")
        else:
            shape = dict(V=_log(rng, 642, 40962), P=rng.choice([1, 2, 4]), map="random")
        return dict(kind="mesh", dtype=rng.choice(["fp32", "bf16"]), B=_log(rng, 1, 8),
                    Ci=_log(rng, 3, 64), Co=_log(rng, 16, 128), K=7, train=rng.random() < 0.75,
                    **shape)
    if kind == "tconv":
        H = _log(rng, 32, 128)
        return dict(kind="tconv", dtype=rng.choice(["fp32", "bf16"]), B=_log(rng, 1, 8),
                    Ci=_log(rng, 8, 64), Co=_log(rng, 3, 64), H=H, W=2 * H + rng.choice([0, 0, 3]),
                    factor=rng.choice([1, 2]), interp=rng.choice(["bilinear", "bispherical"]),
                    train=rng.random() < 0.75)
    if kind in ("max", "avg"):
        H = _log(rng, 48, 512)
        return dict(kind="pool", op=kind, dtype="fp32", B=_log(rng, 1, 4), C=_log(rng, 3, 64), H=H,
                    W=2 * H + rng.choice([0, 0, 0, 1]), stride=rng.choice([1, 2]),
                    map=rng.choice(["latitude", "gnomonic"]),
                    interp=rng.choice(["bilinear", "bispherical", "nearest"]))
    if kind == "resample":
        return dict(kind="resample", op=rng.choice(["resample", "unresample"]), dtype="fp32",
                    B=_log(rng, 1, 4), C=_log(rng, 3, 64), F=_log(rng, 32, 256),
                    interp=rng.choice(["bilinear", "bispherical", "nearest"]))
    return dict(kind="knn", B=rng.choice([1, 1, 2]), D=3, R=_log(rng, 642, 40962),
                Q=_log(rng, 1000, 262144), k=rng.choice([1, 3, 8, 16]))


# ------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _kernel_map(case, dtype):
    """[OH, OW, K, 2] of a spherical kernel on the case's H x W image."""
    H, W, r, stride = case["H"], case["W"], case.get("radius", 1), case.get("stride", 1)
    side = 2 * r + 1
    if case["map"] == "gnomonic":
        return util.get_projection_map((H, W), (side, side), "gnomonic", stride)
    smap = synthetic.latitude_map(H, W, r, dtype=dtype)
    return smap[::stride, ::stride].contiguous().cuda()


def _shuffle_map(g, H, W, dtype):
    """3x3 taps of a grid whose pixels were shuffled, half-way between four pixels; cells
    outside the grid sit at (-0.5, -0.5)."""
    perm = torch.randperm(H * W, generator=g, device="cuda").view(H, W)
    x = torch.full((H + 2, W + 2), -1.0, dtype=dtype, device="cuda")
    y = x.clone()
    x[1:-1, 1:-1], y[1:-1, 1:-1] = (perm % W).to(dtype), (perm // W).to(dtype)
    taps = [torch.stack((x[a:a + H, b:b + W], y[a:a + H, b:b + W]), -1)
            for a in range(3) for b in range(3)]
    return (torch.stack(taps, 2) + 0.5).contiguous()


def _mesh_map(case, g):
    """(indices [1, V, K, P, 2], weights [1, V, K, P]): blends of random vertices, or the
    gnomonic kernel of an icosphere's vertices with barycentric weights."""
    V, K, P = case["V"], case["K"], case["P"]
    if case["map"] == "icosphere":
        order = next(n for n in range(8) if 10 * 4 ** n + 2 == V)
        verts, faces = synthetic.subdivided_icosahedron(order)
        return util.vertex_to_vertex_kernel_map(verts.cuda(), faces.cuda(), 1, K)
    idx = torch.randint(V, (1, V, K, P), generator=g, device="cuda").float()
    smap = torch.stack((idx, torch.zeros_like(idx)), -1).contiguous()
    w = torch.empty(1, V, K, P, device="cuda").exponential_(generator=g)
    return smap, (w / w.sum(-1, keepdim=True)).contiguous()


def _layer(layer, g, fan, dtype):
    """The layer on the GPU, weights and bias from the generator."""
    layer = layer.cuda().to(dtype)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(layer.weight.shape, generator=g, device="cuda") / fan ** 0.5)
        layer.bias.copy_(torch.randn(layer.bias.shape, generator=g, device="cuda") * 0.1)
    return layer


def _sphere(g, B, D, n):
    p = torch.randn(B, D, n, generator=g, device="cuda")
    return (p / p.norm(dim=1, keepdim=True)).contiguous()


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "knn":
        B, D = case["B"], case["D"]
        return dict(kind="knn", ref=_sphere(g, B, D, case["R"]), query=_sphere(g, B, D, case["Q"]),
                    k=case["k"])
    dtype = DTYPES[case["dtype"]]
    map_dtype = torch.float32 if dtype == torch.bfloat16 else dtype
    args, params, interp = (), (), case.get("interp", "nearest")
    if case["kind"] == "conv":
        B, Ci, Co, H, W = (case[n] for n in ("B", "Ci", "Co", "H", "W"))
        K = (2 * case["radius"] + 1) ** 2
        smap = _shuffle_map(g, H, W, dtype) if case["map"] == "shuffle" else \
            _kernel_map(case, map_dtype)
        layer = _layer(nn.MappedConvolution(Ci, Co, K, interp, cache_plan=case["plan"]), g, Ci * K,
                       dtype)
        shape, out, args = (B, Ci, H, W), (B, Co, H, W), (smap,)
    elif case["kind"] == "mesh":
        B, Ci, Co, V, K = (case[n] for n in ("B", "Ci", "Co", "V", "K"))
        layer = _layer(nn.MappedConvolution(Ci, Co, K, interp), g, Ci * K, dtype)
        shape, out, args = (B, Ci, 1, V), (B, Co, 1, V), _mesh_map(case, g)
    elif case["kind"] == "tconv":
        B, Ci, Co, H, W, f = (case[n] for n in ("B", "Ci", "Co", "H", "W", "factor"))
        # the latitude kernel of the fine grid at the positions of the coarse one
        smap = synthetic.latitude_map(f * H, f * W, 1, dtype=map_dtype)
        smap = smap[::f, ::f].contiguous().cuda()
        layer = _layer(nn.MappedTransposedConvolution(Ci, Co, 9, interp), g, Ci * 9, dtype)
        shape, out, args = (B, Ci, H, W), (B, Co, f * H, f * W), (f * H, f * W, smap)
    elif case["kind"] == "pool":
        B, C, H, W = (case[n] for n in ("B", "C", "H", "W"))
        smap = _kernel_map(case, map_dtype)
        layer = nn.MappedMaxPool(9, interp, return_indices=True) if case["op"] == "max" else \
            nn.MappedAvgPool(9, interp)
        shape, out, args = (B, C, H, W), (B, C) + tuple(smap.shape[:2]), (smap,)
    else:
        B, C, F = case["B"], case["C"], case["F"]
        smap = synthetic.cube_to_equirect_map(F, 2 * F, 4 * F, dtype=map_dtype).cuda()
        cube, rect = (B, C, F, 6 * F), (B, C, 2 * F, 4 * F)
        if case["op"] == "resample":
            layer, shape, out, args = nn.Resample(interp), cube, rect, (smap, (2 * F, 4 * F))
        else:
            layer, shape, out, args = nn.Unresample(interp), rect, cube, (smap,)
    if case["kind"] in ("conv", "mesh", "tconv"):
        params = (layer.weight, layer.bias)
    train = case.get("train", True)
    x = torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    gy = torch.randn(out, generator=g, device="cuda", dtype=dtype) if train else None
    return dict(kind=case["kind"], layer=layer, x=x.requires_grad_(train), args=args,
                params=params, gy=gy, train=train)


def run(s):
    if s["kind"] == "knn":
        return util.knn(s["ref"], s["query"], s["k"])
    if not s["train"]:
        with torch.no_grad():
            return s["layer"](s["x"], *s["args"])
    y = s["layer"](s["x"], *s["args"])
    idx = ()
    if isinstance(y, tuple):
        y, idx = y[0], y[1:]
    grads = torch.autograd.grad(y, (s["x"],) + s["params"], s["gy"])
    return (y.detach(),) + idx + grads


# ------------------------------------------------------------------------- measurement
def _conv_flops(c):
    return 6.0 * c["B"] * c["H"] * c["W"] * c["Ci"] * c["Co"] * (2 * c["radius"] + 1) ** 2


def work(case):
    """Every input read once, every output written once; multiply-adds of the products (three
    of them in a training pass), of the taps, or of the distances a grid of cells leaves."""
    kind = case["kind"]
    if kind == "knn":
        B, D, R, Q, k = (case[n] for n in ("B", "D", "R", "Q", "k"))
        return dict(bytes=B * ((R + Q) * D * 4 + Q * k * 12), flops=3.0 * D * B * Q * 4 * k)
    size = SIZE[case["dtype"]]
    map_size = max(size, 4)
    train = case.get("train", True)
    passes = 2 if train else 1
    if kind in ("conv", "mesh", "tconv"):
        B, Ci, Co = case["B"], case["Ci"], case["Co"]
        if kind == "mesh":
            N, M, K, entry = case["V"], case["V"], case["K"], 3 * case["P"]
        else:
            N = case["H"] * case["W"]
            M, K, entry = N, (2 * case.get("radius", 1) + 1) ** 2, 2
            if kind == "tconv":
                M = N * case["factor"] ** 2
        data = passes * size * (B * (Ci * N + Co * M) + Ci * Co * K)
        flops = (6.0 if train else 2.0) * B * N * Ci * Co * K
        return dict(bytes=data + N * K * entry * map_size, flops=flops)
    planes = case["B"] * case["C"]
    if kind == "pool":
        N = case["H"] * case["W"]
        M = -(-case["H"] // case["stride"]) * -(-case["W"] // case["stride"])
        idx = 8 * planes * M if case["op"] == "max" else 0
        return dict(bytes=2 * size * planes * (N + M) + idx + M * 9 * 2 * map_size,
                    flops=2.0 * planes * M * 9 * 8)
    N, M = 6 * case["F"] ** 2, 8 * case["F"] ** 2
    return dict(bytes=2 * size * planes * (N + M) + N * 2 * map_size, flops=2.0 * planes * N * 8)


def tolerance(case):
    """About four times the distance between the 32-bit (bf16) results and the same path in 64
    bits: the longest sums (weight gradients over a million pixels) are off by 1.4e-6 in 2-norm
    and 7e-6 at most, pooled and resampled sums of up to some tens of terms by 8e-8 and 6e-7,
    bf16 results by 2.4e-3 and 1.3e-2 (their own rounding is 1.65e-3).  64-bit sums taken in
    another order differ by 2e-15, but the bias gradient of a single output channel is one sum of
    up to a million terms of both signs: 2e-14 of its value seen.  Whole numbers are equal."""
    if case["kind"] == "knn":
        return "exact"  # the order of a distance's three terms is fixed, ties go by index
    if case["kind"] in ("pool", "resample"):
        return {"rel": 4e-7, "max": 3e-6}
    return {"bf16": {"rel": 1e-2, "max": 0.05}, "fp32": {"rel": 5e-6, "max": 3e-5},
            "fp64": {"rel": 2e-13, "max": 2e-13}}[case["dtype"]]


# ------------------------------------------------------------------- the same in 64 bits
def _corners(smap, weights, H, W, interp):
    """[N, K, corners] element offsets and weights of a map's taps, in 64 bits."""
    x, y = smap.double().unbind(-1)
    if interp == "nearest":
        half = [torch.trunc(v) + torch.where((v - torch.trunc(v)).abs() >= 0.5, v.sign(), 0 * v)
                for v in (x, y)]
        cols, rows, wts = [half[0]], [half[1]], [torch.ones_like(x)]
    else:
        x1, y1 = x.floor(), y.floor()
        cols, rows = [x1, x1 + 1] * 2, [y1, y1, y1 + 1, y1 + 1]
        A, B, C, D = y1 + 1 - y, x1 + 1 - x, x - x1, y - y1
        wts = [A * B, A * C, D * B, D * C]
        if interp == "bispherical":
            cols = [c % W for c in cols]
    off, wt = [], []
    for c, r, a in zip(cols, rows, wts):
        inside = (c >= 0) & (c < W) & (r >= 0) & (r < H)
        off.append(torch.where(inside, r * W + c, 0 * c).long())
        wt.append(torch.where(inside, a if weights is None else a * weights.double(), 0 * a))
    off, wt = torch.stack(off, -1), torch.stack(wt, -1)
    if weights is not None:  # [..., P, corners]: all of them belong to the same tap
        off, wt = off.flatten(-2), wt.flatten(-2)
    n = smap.shape[0] * smap.shape[1]
    return off.reshape(n, -1, off.shape[-1]), wt.reshape(n, -1, off.shape[-1])


def _gather(plane, off, wt):
    """[C, N] samples of [C, HW] planes at [N, corners]."""
    return sum(plane[:, off[:, i]] * wt[:, i] for i in range(off.shape[1]))


def _scatter(plane, values, off, wt):
    for i in range(off.shape[1]):
        plane.index_add_(1, off[:, i], values * wt[:, i])


def exact(case, seed):
    if case["kind"] == "knn" or work(case)["flops"] > 2e12:
        return None  # whole numbers beside distances of fixed order; over 20 seconds
    s = prepare(case, seed)
    kind, train, smap = case["kind"], s["train"], s["args"][0]
    weights, (H, W) = None, s["x"].shape[2:]
    x = s["x"].detach().double().flatten(2)
    gy = s["gy"].double().flatten(2) if train else [None] * len(x)
    if kind == "tconv":
        H, W, smap = s["args"]
    elif kind == "mesh":
        weights = s["args"][1]
    elif case.get("op") == "resample":
        H, W = s["args"][1]
    off, wt = _corners(smap, weights, H, W, case.get("interp", "nearest"))
    taps = range(off.shape[1])
    plane = lambda c: torch.zeros(c, H * W, dtype=torch.float64, device="cuda")
    if kind in ("pool", "resample"):
        y, gx = [], []
        for xb, gb in zip(x, gy):
            if case.get("op") == "resample":
                y.append(plane(len(xb)))
                _scatter(y[-1], xb, off[:, 0], wt[:, 0])
                gx.append(_gather(gb, off[:, 0], wt[:, 0]))
                continue
            cols = (_gather(xb, off[:, k], wt[:, k]) for k in taps)
            if case.get("op") == "max":
                best = next(cols)
                for c in cols:
                    best = torch.maximum(best, c)
                y.append(best)
                continue
            y.append(sum(cols) / len(taps))
            gx.append(plane(len(xb)))
            for k in taps:
                _scatter(gx[-1], gb / len(taps), off[:, k], wt[:, k])
        shape = s["gy"].shape
        y = torch.stack(y).view(shape)
        # which of two taps within rounding of each other wins is not a matter of precision
        return (y, None, None) if case.get("op") == "max" else \
            (y, torch.stack(gx).view(s["x"].shape))
    w, bias = (p.detach().double() for p in s["params"])
    y, gx, gw = [], [], torch.zeros_like(w)
    for xb, gb in zip(x, gy):
        if kind == "tconv":
            y.append(plane(w.shape[1]) + bias[:, None])
            gx.append(torch.zeros_like(xb))
            for k in taps:
                _scatter(y[-1], w[:, :, k].t() @ xb, off[:, k], wt[:, k])
                if train:
                    col = _gather(gb, off[:, k], wt[:, k])
                    gx[-1] += w[:, :, k] @ col
                    gw[:, :, k] += xb @ col.t()
            continue
        y.append(bias[:, None].repeat(1, len(off)))
        gx.append(plane(len(xb)))
        for k in taps:
            col = _gather(xb, off[:, k], wt[:, k])
            y[-1] += w[:, :, k] @ col
            if train:
                gw[:, :, k] += gb @ col.t()
                _scatter(gx[-1], w[:, :, k].t() @ gb, off[:, k], wt[:, k])
    y = torch.stack(y)
    if not train:
        return y.view(len(y), y.shape[1], *((H, W) if kind == "tconv" else smap.shape[:2]))
    return (y.view(s["gy"].shape), torch.stack(gx).view(s["x"].shape), gw, gy.sum((0, 2)))
