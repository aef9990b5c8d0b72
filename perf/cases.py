"""Performance cases of the sparse-convolution framework.

Every case is work that a program hands to the public entry points
(``sparsetriton_amd``): convolution layers in training and inference, the
residual block, the backbone, pooling and upsampling.  ``listed()`` names the
cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` builds
what the program has in hand before the call, ``run`` is one pass, ``exact``
the same pass in float64 from plain torch.

Case fields
  family     "conv" (one layer), "block" (SparseResBlock, training), "net"
             (SparseResNet21D, inference), "pool" (pooling + upsampling, training)
  voxels     coordinate set: "lidar" (ground rings and box faces of a spinning
             scanner in 1440 x 1440 x 41, ~4.7 of 27 neighbours occupied),
             "indoor" (two-voxel-thick walls and floors in a cube, ~17 of 27),
             "uniform" (random voxels of a 64^3 box, nearly isolated)
  n, batch   rows (over all samples) and samples
  op, k, s   conv: "subm", "strided" (padding (k - 1) // 2) or "transposed"
             (no padding), kernel size and stride
  cin, cout  channels;  dtype  "f32", "bf16", "f16" (features and weights)
  algo       conv: "map" (precomputed kernel map) or "fly" (in-GEMM lookups)
  train      conv: forward and backward, or inference
  fresh      conv: the coordinates are new in every pass, so the pass builds the
             index, map and plans (the first layer of a stage); otherwise the
             coordinate set's maps are there already (its later layers)
  xgrad      conv: the features need a gradient (not so for a first layer)
"""

import math
import random
import zlib

import torch

import sparsetriton_amd as st
from sparsetriton_amd import config, nn

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ESZ = {"f32": 4, "bf16": 2, "f16": 2}
ALGOS = {"map": config.ConvAlgo.PrecomputedNeighborGEMM, "fly": config.ConvAlgo.ImplicitHashFlyGEMM}
LIDAR_SHAPE = (1440, 1440, 41)
STAGES = ((3, 16, 1), (3, 32, 2), (3, 64, 2), (3, 128, 2), (1, 128, 2))  # blocks, channels, stride


def _conv(name=None, **kw):
    c = {"family": "conv", "voxels": "lidar", "n": 0, "batch": 1, "op": "subm", "k": 3, "s": 1, "cin": 64, "cout": 64,
         "dtype": "f32", "algo": "map", "train": True, "fresh": False, "xgrad": True, "bias": False}
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The reference test's and CPU baseline's layer size: 4,096 voxels, where launches and host work count.
        _conv("subm_4k_16x32_f32_train", voxels="uniform", n=4096, batch=2, cin=16, cout=32, bias=True),
        # The benchmark's headline layer: a 64-channel backbone layer on four LiDAR sweeps, default fp32.
        _conv("subm_lidar_64_f32_train", n=470_532, batch=4),
        # The same layer in the 16-bit type most training runs use.
        _conv("subm_lidar_64_bf16_train", n=470_532, batch=4, dtype="bf16"),
        # A stage's downsampling layer (64 -> 128, stride 2), fp32 training.
        _conv("strided_64x128_f32_train", n=470_532, batch=4, op="strided", s=2, cout=128),
        # A decoder's upsampling layer on new coordinates, inference: the output-coordinate and map
        # build with the convolution, the largest output.
        _conv("transposed_128x64_bf16_infer", n=240_001, batch=2, op="transposed", s=2, cin=128, dtype="bf16", train=False,
              fresh=True),
        # A wide layer on a large indoor scan: the contraction-bound end, forward and backward.
        _conv("subm_indoor_1m_128_bf16_train", voxels="indoor", n=1_000_000, cin=128, cout=128, dtype="bf16"),
        # The map-free algorithm, which memory-limited programs choose, in fp16.
        _conv("fly_indoor_300k_64x128_f16_train", voxels="indoor", n=300_007, cin=64, cout=128, dtype="f16", algo="fly"),
        # The network's entry layer on a new batch of sweeps: index, map and plans built in the pass,
        # point features 4 -> 16, weight gradient only.
        _conv("entry_lidar_4x16_f32_train", n=470_532, batch=4, cin=4, cout=16, fresh=True, xgrad=False, bias=True),
        # A segmentation head's layer on one sweep, inference: odd row count, 20 classes.
        _conv("head_lidar_32x20_f16_infer", n=50_001, cin=32, cout=20, dtype="f16", train=False, bias=True),
        # A residual block of the backbone's second stage in training: convolutions, per-sample batch
        # norms, ReLU and the residual add, forward and backward.
        {"name": "block_lidar_32_f32_train", "family": "block", "voxels": "lidar", "n": 250_003, "batch": 4, "cin": 32,
         "dtype": "f32"},
        # The whole backbone on one new sweep: the latency of a deployed detector's 3-D part.
        {"name": "resnet21d_sweep_bf16_infer", "family": "net", "voxels": "lidar", "n": 117_000, "batch": 1, "cin": 4,
         "dtype": "bf16"},
        # An encoder-decoder's pooling and upsampling pair in training.
        {"name": "pool_up_lidar_64_bf16_train", "family": "pool", "voxels": "lidar", "n": 200_001, "batch": 2, "cin": 64,
         "k": 2, "s": 2, "mode": "max", "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """One more case of the listed cases' ranges; never more work than the largest listed one."""
    kind = rng.choice(["train"] * 4 + ["infer", "entry", "strided", "strided", "transposed", "fly", "block", "net", "pool"])
    dtype = rng.choice(["f32", "f32", "bf16", "bf16", "f16"])
    ch = [16, 32, 64, 128]
    voxels = rng.choice(["lidar", "lidar", "indoor", "uniform"])
    sweeps = rng.choice([1, 2, 4])
    hi = {"lidar": 117_000 * sweeps, "indoor": 900_000, "uniform": 200_000}[voxels]
    batch = {"lidar": sweeps, "indoor": 1, "uniform": 2}[voxels]
    if kind == "train":
        return _conv(voxels=voxels, n=_log(rng, 2000, hi), batch=batch, cin=rng.choice(ch), cout=rng.choice(ch + [20]),
                     dtype=dtype if voxels != "indoor" else "bf16", bias=rng.random() < 0.5)
    if kind == "infer":
        return _conv(voxels=voxels, n=_log(rng, 2000, hi), batch=batch, cin=rng.choice(ch), cout=rng.choice([16, 20, 32, 64]),
                     dtype=dtype, train=False, bias=True)
    if kind == "entry":
        return _conv(n=_log(rng, 5000, 117_000 * sweeps), batch=sweeps, cin=rng.choice([4, 16]),
                     cout=rng.choice([16, 32]), dtype=dtype, fresh=True, xgrad=False, bias=True)
    if kind == "strided":
        return _conv(n=_log(rng, 4000, 117_000 * sweeps), batch=sweeps, op="strided", s=2,
                     k=rng.choice([3, 3, 2]), cin=rng.choice([16, 32, 64]), cout=rng.choice([32, 64, 128]), dtype=dtype,
                     train=rng.random() < 0.6, fresh=False)
    if kind == "transposed":
        return _conv(n=_log(rng, 4000, 60_000 * sweeps), batch=sweeps, op="transposed", s=2, cin=rng.choice([64, 128]),
                     cout=rng.choice([32, 64]), dtype=rng.choice(["bf16", "f16"]), train=False, fresh=True)
    if kind == "fly":
        return _conv(voxels="indoor", n=_log(rng, 10_000, 300_000), cin=rng.choice([64, 128]), cout=rng.choice([64, 128]),
                     dtype=rng.choice(["bf16", "f16"]), algo="fly")
    if kind == "block":
        return {"family": "block", "voxels": "lidar", "n": _log(rng, 5000, 62_000 * sweeps), "batch": sweeps,
                "cin": rng.choice([16, 32, 64]), "dtype": "f32"}
    if kind == "net":
        return {"family": "net", "voxels": "lidar", "n": _log(rng, 20_000, 100_000), "batch": min(sweeps, 2), "cin": 4,
                "dtype": rng.choice(["bf16", "f16"])}
    return {"family": "pool", "voxels": "lidar", "n": _log(rng, 5000, 100_000 * sweeps), "batch": sweeps,
            "cin": rng.choice([16, 32, 64]), "k": 2, "s": 2, "mode": rng.choice(["max", "avg"]), "dtype": dtype}


# ------------------------------------------------------------- inputs

def _gens(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return random.Random(seed), g


def _lidar(case, seed):
    """(n, 4) int16 coordinates sorted by (b, x, y, z): per sample the voxels nearest to the scanner.
    The scenes belong to the case; the seed moves them by multiples of 16 voxels, swaps x and y and
    reorders the samples, so every seed has other coordinates but the same row counts in every layer."""
    n, batch = case["n"], case["batch"]
    rng, g = _gens(zlib.crc32(f"{n} {batch}".encode()))
    pick = random.Random(seed)
    swap = pick.random() < 0.5
    order = pick.sample(range(batch), batch)
    X, Y, Z = LIDAR_SHAPE
    parts = [None] * batch
    for b in range(batch):
        want = n // batch + (1 if b < n % batch else 0)
        dx, dy = 16 * pick.randint(-3, 3), 16 * pick.randint(-3, 3)
        ph = [rng.uniform(0, 2 * math.pi) for _ in range(4)]
        f = [rng.uniform(60, 160) for _ in range(4)]
        cx, cy = X / 2, Y / 2

        def height(x, y):
            v = Z * 0.3 + 2.5 * torch.sin(x / f[0] + ph[0]) + 2.0 * torch.sin(y / f[1] + ph[1])
            v = v + 1.5 * torch.sin((x + y) / f[2] + ph[2]) + torch.sin((x - y) / f[3] + ph[3])
            return v.round().clamp(0, Z - 1)

        # ground rings whose radii grow geometrically
        rad = 12.0 * 1.062 ** torch.arange(70, device="cuda", dtype=torch.float64)
        rad = rad[rad < 660]
        th = torch.arange(2600, device="cuda", dtype=torch.float64) * (2 * math.pi / 2600)
        x = (cx + rad[:, None] * torch.cos(th)).round().reshape(-1)
        y = (cy + rad[:, None] * torch.sin(th)).round().reshape(-1)
        pts = [torch.stack([x, y, height(x, y)], 1)]
        # the two visible faces of 260 boxes, 60 % of their voxels returned
        box = torch.rand(260, 5, generator=g, device="cuda", dtype=torch.float64)
        r, a = 15 + box[:, 0] * 600, box[:, 1] * 2 * math.pi
        x0, y0 = (cx + r * torch.cos(a)).floor(), (cy + r * torch.sin(a)).floor()
        w, h = (8 + box[:, 2:4] * 32).floor(), (4 + box[:, 4] * 10).floor()
        z0 = height(x0, y0)
        u = torch.arange(40, device="cuda", dtype=torch.float64)
        v = torch.arange(14, device="cuda", dtype=torch.float64)
        for face in (0, 1):
            along = u[None, :, None].expand(260, 40, 14)
            up = v[None, None, :].expand(260, 40, 14)
            ok = (along < w[:, face, None, None]) & (up < h[:, None, None]) & (z0[:, None, None] + up < Z)
            ok &= torch.rand(260, 40, 14, generator=g, device="cuda") < 0.6
            px = x0[:, None, None] + (along if face else 0 * along)
            py = y0[:, None, None] + (0 * along if face else along)
            pts.append(torch.stack([px[ok], py[ok], (z0[:, None, None] + up)[ok]], 1))
        p = torch.cat(pts).long()
        key = torch.unique((p[:, 0] * Y + p[:, 1]) * Z + p[:, 2])
        x, y, z = key // (Y * Z), key // Z % Y, key % Z
        if key.numel() < want:
            raise ValueError(f"the scene holds {key.numel()} voxels, {want} asked for")
        near = torch.sort((x - cx) ** 2 + (y - cy) ** 2, stable=True).indices[:want]
        x, y, z = x[near] + dx, y[near] + dy, z[near]
        if swap:
            x, y = y, x
        key = ((x * Y + y) * Z + z).sort().values
        parts[order[b]] = torch.stack([torch.full_like(key, order[b]), key // (Y * Z), key // Z % Y, key % Z], 1)
    return torch.cat(parts).to(torch.int16)


def _indoor(rng, g, n):
    """(n, 4) int16 coordinates of two-voxel-thick axis-aligned planes in a cube."""
    S = max(32, min(256, int(round((n / 1_000_000) ** (1 / 3) * 256))))
    grid = torch.zeros((S, S, S), dtype=torch.bool, device="cuda")
    while True:
        for _ in range(4):
            axis, pos = rng.randrange(3), rng.randrange(S - 2)
            lo = [rng.randrange(S // 2) for _ in range(2)]
            hi = [min(S, v + rng.randrange(S // 3, S)) for v in lo]
            sl = [slice(lo[0], hi[0]), slice(lo[1], hi[1])]
            sl.insert(axis, slice(pos, pos + 2))
            grid[tuple(sl)] = True
        if int(grid.sum()) >= n:
            break
    c = grid.nonzero()
    keep = torch.randperm(c.shape[0], generator=g, device="cuda")[:n].sort().values
    c = c[keep]
    return torch.cat([torch.zeros_like(c[:, :1]), c], 1).to(torch.int16), (S, S, S)


def _coords(case, seed, rng, g):
    n, B = case["n"], case["batch"]
    if case["voxels"] == "lidar":
        return _lidar(case, seed), LIDAR_SHAPE
    if case["voxels"] == "indoor":
        return _indoor(rng, g, n)
    lin = torch.randperm(B * 64 ** 3, generator=g, device="cuda")[:n].sort().values
    c = torch.stack([lin // 64 ** 3, lin // 4096 % 64, lin // 64 % 64, lin % 64], 1)
    return c.to(torch.int16), (64, 64, 64)


def _rand(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _inputs(case, seed):
    """Coordinates, features and the layers' parameters, all from the seed."""
    rng, g = _gens(seed)
    dt = DTYPES[case["dtype"]]
    coords, shape = _coords(case, seed, rng, g)
    d = {"coords": coords, "shape": shape, "feats": _rand(g, coords.shape[0], case["cin"], dtype=dt), "g": g}

    def weight(k3, ci, co):
        bound = 1 / math.sqrt(ci * k3)
        return ((torch.rand(k3, ci, co, generator=g, device="cuda") * 2 - 1) * bound).to(dt), \
               ((torch.rand(co, generator=g, device="cuda") * 2 - 1) * bound).to(dt)

    def norm(c):
        return (0.5 + torch.rand(c, generator=g, device="cuda"), _rand(g, c) * 0.1,
                _rand(g, c) * 0.05, 0.05 + 0.1 * torch.rand(c, generator=g, device="cuda"))

    if case["family"] == "conv":
        d["w"], b = weight(case["k"] ** 3, case["cin"], case["cout"])
        d["b"] = b if case["bias"] else None
    elif case["family"] == "block":
        C = case["cin"]
        d["convs"] = [weight(27, C, C) for _ in range(2)]
        d["norms"] = [norm(C) for _ in range(2)]
    elif case["family"] == "net":
        d["convs"], d["norms"], ci = [], [], case["cin"]
        for blocks, co, _ in STAGES:
            for i in range(2 * blocks - 1):
                d["convs"].append(weight(27, ci, co))
                d["norms"].append(norm(co))
                ci = co
    return d


def _load(module, d, dtype):
    """Puts the inputs' parameters into a module's convolutions and batch norms, in module order."""
    convs = [m for m in module.modules() if isinstance(m, nn.SparseConv3DBase)]
    norms = [m for m in module.modules() if isinstance(m, nn.SparseBatchNorm)]
    assert len(convs) == len(d["convs"]) and len(norms) == len(d["norms"])
    with torch.no_grad():
        for m, (w, b) in zip(convs, d["convs"]):
            m.to(dtype)  # batch norms stay fp32
            m.weight.copy_(w)
            m.bias.copy_(b)
        for m, (w, b, mean, var) in zip(norms, d["norms"]):
            for dst, src in ((m.weight, w), (m.bias, b), (m.running_mean, mean), (m.running_var, var)):
                dst.copy_(src)


def prepare(case, seed):
    d = _inputs(case, seed)
    g, dt = d.pop("g"), DTYPES[case["dtype"]]
    s = {"case": dict(case), "coords": d["coords"], "shape": d["shape"], "batch": case["batch"], "feats": d["feats"]}
    if case["family"] == "net":
        model = nn.SparseResNet21D(in_channels=case["cin"]).cuda().eval()
        _load(model, d, dt)
        s["model"] = model
        return s
    x = st.SparseTensor(d["feats"], d["coords"], spatial_shape=d["shape"], batch_size=case["batch"])
    if case["family"] == "pool":
        s["feats"].requires_grad_(True)
        s["x"] = x
        with torch.no_grad():
            n_out = nn.functional.sparse_pooling(x, case["k"], 0, case["s"], case["mode"]).F.shape[0]
        s["gp"] = _rand(g, n_out, case["cin"], dtype=dt)
        s["gu"] = _rand(g, n_out * 8, case["cin"], dtype=dt)
        return s
    config.set_conv_algo(ALGOS[case.get("algo", "map")])
    if case["family"] == "block":
        block = nn.SparseResBlock(case["cin"], case["cin"], 3).cuda().train()
        _load(block, d, dt)
        s["feats"].requires_grad_(True)
        s.update(block=block, x=x, gy=_rand(g, *s["feats"].shape, dtype=dt))
        with torch.enable_grad():
            block.main[0](x)  # the coordinate set's map, which an earlier layer of the stage has built
        return s
    kind = {"subm": nn.SubMConv3D, "strided": nn.SparseConv3D, "transposed": nn.SparseConvTransposed3D}[case["op"]]
    pad = {"padding": (case["k"] - 1) // 2} if case["op"] == "strided" else {}
    conv = kind(case["cin"], case["cout"], case["k"], stride=case["s"], bias=case["bias"], **pad).cuda().to(dt)
    with torch.no_grad():
        conv.weight.copy_(d["w"])
        if case["bias"]:
            conv.bias.copy_(d["b"])
    s["conv"] = conv
    if case["train"] and case["xgrad"]:
        s["feats"].requires_grad_(True)
    if not case["fresh"]:
        s["x"] = x
        with torch.set_grad_enabled(case["train"]):
            n_out = conv(x).F.shape[0]  # an earlier layer of the stage has built the map
    else:
        n_out = case["n"]  # (fresh training cases are submanifold)
    if case["train"]:
        s["gy"] = _rand(g, n_out, case["cout"], dtype=dt)
    return s


# --------------------------------------------------------------- a pass

def run(state):
    case = state["case"]
    fam = case["family"]
    if fam == "pool":
        x = state["x"]
        low = nn.functional.sparse_pooling(x, case["k"], 0, case["s"], case["mode"])
        up = nn.functional.sparse_upsample(low, 2)
        (dx,) = torch.autograd.grad([low.F, up.F], [state["feats"]], [state["gp"], state["gu"]])
        return {"low": low.F.detach(), "low_c": low.C, "up": up.F.detach(), "up_c": up.C, "dx": dx}
    config.set_conv_algo(ALGOS[case.get("algo", "map")])
    if fam == "block":
        block = state["block"]
        out = block(state["x"])
        params = list(block.parameters())
        grads = list(torch.autograd.grad(out.F, [state["feats"]] + params, state["gy"]))
        # the gradients of the biases before a batch norm are zero but for rounding: computed, nothing to compare
        del grads[6], grads[2]
        running = [t for m in (block.main[1], block.main[4]) for t in (m.running_mean, m.running_var)]
        return {"y": out.F.detach(), "grads": grads, "running": running}
    if fam == "net":
        with torch.no_grad():
            x = st.SparseTensor(state["feats"], state["coords"], spatial_shape=state["shape"], batch_size=state["batch"])
            outs = state["model"](x)
        return {"y": [o.F for o in outs], "c": [o.C for o in outs[1:]]}
    conv = state["conv"]
    if case["fresh"]:
        x = st.SparseTensor(state["feats"], state["coords"], spatial_shape=state["shape"], batch_size=state["batch"])
    else:
        x = state["x"]
    if not case["train"]:
        with torch.no_grad():
            out = conv(x)
        return {"y": out.F, "c": out.C} if case["op"] != "subm" else {"y": out.F}
    out = conv(x)
    wrt = ([state["feats"]] if case["xgrad"] else []) + list(conv.parameters())
    grads = torch.autograd.grad(out.F, wrt, state["gy"])
    return {"y": out.F.detach(), "grads": list(grads)}


# ------------------------------------------------------------- its work

PAIRS = {"lidar": 4.7, "indoor": 17.0}  # mean occupied sites of a voxel's 3 x 3 x 3 neighbourhood


def _pairs(case):
    """(output rows, pairs) per input row, typical of the coordinate set."""
    if case["voxels"] == "uniform":
        return 1.0, 1 + 26 * case["n"] / (case["batch"] * 64 ** 3)
    per = PAIRS[case["voxels"]]
    if case.get("op") == "strided":
        return (1.0, 27 / 8) if case["k"] == 3 else (0.5, 1.0)
    if case.get("op") == "transposed":
        return 18.0, 27.0
    return 1.0, per


def work(case):
    n, e = case["n"], ESZ[case["dtype"]]
    if case["family"] == "pool":
        C, out = case["cin"], 0.5 * n
        # pooled rows and their children written, the features and both gradients read, dx written
        return {"bytes": e * C * (n + out + 8 * out + out + 8 * out + n + n) + 8 * (n + out + 8 * out), "flops": 0.0}
    if case["family"] == "block":
        C, p = case["cin"], PAIRS["lidar"] * n
        conv = 3 * (2 * n * C * e + 8 * p + 27 * C * C * e)
        norm = 8 * n * C * e
        return {"bytes": 2 * conv + 2 * norm, "flops": 2 * 6.0 * p * C * C}
    if case["family"] == "net":
        rows, ci, by, fl = float(n), case["cin"], 8.0 * n, 0.0
        for (blocks, co, s), grow, per in zip(STAGES, (1, 1.02, 0.55, 0.5, 0.4), (4.7, 11.3, 13.3, 15.0, 17.0)):
            src, rows = rows, rows * grow
            for i in range(2 * blocks - 1):
                p = (27 / 8 * src) if (i == 0 and s > 1) else per * rows
                by += e * ((src if i == 0 else rows) * ci + rows * co + 27 * ci * co)
                fl += 2 * p * ci * co
                ci = co
            by += 8 * rows
        return {"bytes": by, "flops": fl}
    grow, per = _pairs(case)
    p, out, ci, co = per * n, grow * n, case["cin"], case["cout"]
    passes = 1 if not case["train"] else (3 if case["xgrad"] else 2)
    by = passes * (e * (n * ci + out * co + case["k"] ** 3 * ci * co) + (8 * p if not case["fresh"] else 0))
    return {"bytes": by + (8 * n + 8 * out if case["fresh"] else 0), "flops": passes * 2.0 * p * ci * co}


def tolerance(case):
    fam, dt = case["family"], case["dtype"]
    if fam == "pool":
        # values are moved or averaged over at most eight rows and rounded once
        return {"rel": {"f32": 1e-6, "bf16": 1e-2, "f16": 1.5e-3}[dt]}
    if fam == "block":
        return {"rel": 1.2e-2}  # ReLU decisions within rounding of zero: a share f of them moves the gradients by sqrt(f)
    if fam == "net":
        return {"rel": {"bf16": 2.5e-2, "f16": 4e-3}[dt]}
    return {"rel": {"f32": 2e-5, "bf16": 7e-3, "f16": 9e-4}[dt]}


# --------------------------------------------- the same pass in float64

def _base(k):
    i = torch.arange(k, device="cuda") - k // 2
    return torch.stack(torch.meshgrid(i, i, i, indexing="ij"), -1).reshape(-1, 3)


def _key(c):
    return ((c[..., 0] * 8192 + c[..., 1] + 64) * 8192 + c[..., 2] + 64) * 8192 + c[..., 3] + 64


def _out_coords(c, shape, k, s, p, transposed):
    """Output coordinates in order of their first candidate (rows outer, offsets inner), and the shape."""
    base = _base(k)
    if transposed:
        t, new = base - p + (k - 1) // 2, [(v - 1) * s + (k - 1) - 2 * p + 1 for v in shape]
        cand = c[:, None, 1:] * s + t
        ok = torch.ones(cand.shape[:2], dtype=torch.bool, device="cuda")
    else:
        t, new = -base + p - (k - 1) // 2, [(v - (k - 1) + 2 * p - 1) // s + 1 for v in shape]
        cand = c[:, None, 1:] + t
        ok = (cand % s == 0).all(-1)
        cand = torch.div(cand, s, rounding_mode="floor")
    ok &= ((cand >= 0) & (cand < torch.tensor(new, device="cuda"))).all(-1)
    cand = torch.cat([c[:, None, :1].expand(-1, k ** 3, 1), cand], 2)[ok]
    uniq, inv = torch.unique(_key(cand), return_inverse=True)
    first = torch.full((uniq.numel(),), cand.shape[0], dtype=torch.long, device="cuda")
    first.scatter_reduce_(0, inv, torch.arange(cand.shape[0], device="cuda"), "amin")
    return cand[first.sort().values], tuple(new)


def _map64(c_in, c_out, shape, k, s, p, transposed):
    """Per offset the (input rows, output rows) pairs."""
    keys, order = _key(c_in).sort()
    base, out = _base(k), []
    lim = torch.tensor(shape, device="cuda")
    for j in range(k ** 3):
        if transposed:
            q = c_out[:, 1:] - (base[j] - p + (k - 1) // 2)
            ok = (q % s == 0).all(-1)
            q = torch.div(q, s, rounding_mode="floor")
        else:
            q = c_out[:, 1:] * s + base[j] - p + (k - 1) // 2
            ok = torch.ones(q.shape[0], dtype=torch.bool, device="cuda")
        ok &= ((q >= 0) & (q < lim)).all(-1)
        qk = _key(torch.cat([c_out[:, :1], q], 1))
        pos = torch.searchsorted(keys, qk).clamp_(max=keys.numel() - 1)
        o = (ok & (keys[pos] == qk)).nonzero()[:, 0]
        out.append((order[pos[o]], o))
    return out


class _Conv64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, pairs, n_out):
        ctx.save_for_backward(x, w)
        ctx.pairs = pairs
        y = torch.zeros((n_out, w.shape[2]), dtype=torch.float64, device="cuda")
        for j, (i, o) in enumerate(pairs):
            if i.numel():
                y.index_add_(0, o, x[i] @ w[j])
        return y

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dx, dw = torch.zeros_like(x), torch.zeros_like(w)
        for j, (i, o) in enumerate(ctx.pairs):
            if i.numel():
                g = dy[o]
                dx.index_add_(0, i, g @ w[j].t().contiguous())
                dw[j] = x[i].t().contiguous() @ g
        return dx, dw, None, None


def _norm_train64(y, rows, B, w, b):
    mean, var = [], []
    out = torch.empty_like(y)
    for s in range(B):
        sel = (rows == s).nonzero()[:, 0]
        m, v = y[sel].mean(0), y[sel].var(0, unbiased=False)
        out = out.index_copy(0, sel, (y[sel] - m) / torch.sqrt(v + 1e-5) * w + b)
        mean.append(m.detach())
        var.append(v.detach())
    return out, torch.stack(mean).mean(0), torch.stack(var).mean(0)


def exact(case, seed):
    d = _inputs(case, seed)
    g, dt = d.pop("g"), DTYPES[case["dtype"]]
    c, x = d["coords"].long(), d["feats"].double()
    fam = case["family"]
    if fam == "pool":
        k, s = case["k"], case["s"]
        cell = torch.cat([c[:, :1], torch.div(c[:, 1:] - k // 2, s, rounding_mode="floor")], 1)
        _, inv = torch.unique(_key(cell), return_inverse=True)
        n_out = int(inv.max()) + 1
        gp, gu = _rand(g, n_out, case["cin"], dtype=dt), _rand(g, n_out * 8, case["cin"], dtype=dt)
        low_c = torch.zeros((n_out, 4), dtype=torch.long, device="cuda").index_copy_(0, inv, cell)
        idx = inv[:, None].expand(-1, x.shape[1])
        total = gp.double() + gu.double().view(n_out, 8, -1).sum(1)
        if case["mode"] == "max":
            low = torch.full((n_out, x.shape[1]), -math.inf, dtype=torch.float64, device="cuda")
            low.scatter_reduce_(0, idx, x, "amax")
            dx = torch.where(x == low[inv], total[inv], torch.zeros((), dtype=torch.float64, device="cuda"))
        else:
            cnt = torch.bincount(inv, minlength=n_out).double()[:, None]
            low = torch.zeros((n_out, x.shape[1]), dtype=torch.float64, device="cuda").index_add_(0, inv, x) / cnt
            dx = (total / cnt)[inv]
        off = _base(2) + 1
        up_c = torch.cat([low_c[:, None, :1].expand(-1, 8, 1), low_c[:, None, 1:] * 2 + off], 2).reshape(-1, 4)
        return {"low": low, "low_c": low_c.to(torch.int16), "up": low.repeat_interleave(8, 0), "up_c": up_c.to(torch.int16),
                "dx": dx}
    if fam == "block":
        pairs = _map64(c, c, d["shape"], 3, 1, 1, False)
        p = [t.double().requires_grad_(True) for i in range(2) for t in d["convs"][i] + d["norms"][i][:2]]
        w1, b1, nw1, nb1, w2, b2, nw2, nb2 = p
        x.requires_grad_(True)
        n = x.shape[0]
        running = []

        def norm(y, i, w, b):
            out, mean, var = _norm_train64(y, c[:, 0], case["batch"], w, b)
            running.extend([0.9 * d["norms"][i][2].double() + 0.1 * mean, 0.9 * d["norms"][i][3].double() + 0.1 * var])
            return out

        h = torch.relu(norm(_Conv64.apply(x, w1, pairs, n) + b1, 0, nw1, nb1))
        y = torch.relu(norm(_Conv64.apply(h, w2, pairs, n) + b2, 1, nw2, nb2) + x)
        gy = _rand(g, *x.shape, dtype=dt).double()
        grads = list(torch.autograd.grad(y, [x] + p, gy))
        del grads[6], grads[2]
        return {"y": y.detach(), "grads": grads, "running": running}
    if fam == "net":
        shape, ys, cs, at, first = d["shape"], [], [], 0, True

        def conv_norm(x, pairs, n, res=None, relu=True):
            nonlocal at
            (w, b), (nw, nb, mean, var) = d["convs"][at], d["norms"][at]
            at += 1
            y = _Conv64.apply(x, w.double(), pairs, n) + b.double()
            y = (y - mean.double()) / torch.sqrt(var.double() + 1e-5) * nw.double() + nb.double()
            return torch.relu(y if res is None else y + res)

        with torch.no_grad():
            for blocks, co, s in STAGES:
                if s > 1:
                    co_, new = _out_coords(c, shape, 3, s, 1, False)
                    pairs = _map64(c, co_, shape, 3, s, 1, False)
                    c, shape = co_, new
                    x = conv_norm(x, pairs, c.shape[0])
                pairs = _map64(c, c, shape, 3, 1, 1, False)
                if s == 1:
                    x = conv_norm(x, pairs, c.shape[0])
                for _ in range(blocks - 1):
                    h = conv_norm(x, pairs, c.shape[0])
                    x = conv_norm(h, pairs, c.shape[0], res=x)
                ys.append(x)
                if not first:
                    cs.append(c.to(torch.int16))
                first = False
        return {"y": ys, "c": cs}
    k, s, tr = case["k"], case["s"], case["op"] == "transposed"
    p = 0 if tr else (k - 1) // 2
    co_ = c if case["op"] == "subm" else _out_coords(c, d["shape"], k, s, p, tr)[0]
    pairs = _map64(c, co_, d["shape"], k, s, p, tr)
    w = d["w"].double()
    y = _Conv64.apply(x, w, pairs, co_.shape[0])
    if d["b"] is not None:
        y = y + d["b"].double()
    if not case["train"]:
        return {"y": y} if case["op"] == "subm" else {"y": y, "c": co_.to(torch.int16)}
    gy = _rand(g, co_.shape[0], case["cout"], dtype=dt).double()
    grads = []
    ctx = type("Ctx", (), {"saved_tensors": (x, w), "pairs": pairs})
    dx, dw, _, _ = _Conv64.backward(ctx, gy)
    if case["xgrad"]:
        grads.append(dx)
    grads.append(dw)
    if d["b"] is not None:
        grads.append(gy.sum(0))
    return {"y": y, "grads": grads}
