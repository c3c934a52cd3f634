"""The sparse hot path as a user's program calls it: which calls, at which sizes, on
which inputs, and what they compute in 64 bits.

A case is one public entry point at one size. ``kind`` says which:

* ``layer``: one ``SubMConv3d`` on a coordinate set whose kernel map is cached, as every
  layer of a network but the first of its level runs.
* ``first``: the same module on a coordinate set seen for the first time: kernel map,
  tile plan and convolution.
* ``strided``: ``SparseConv3d`` (2x2x2, stride 2) and its ``SparseInverseConv3d``.
* ``block``: the adaLN residual block (norm + modulation, convolution + SiLU,
  convolution + residual).
* ``resblock3d``: the transformer's ``SparseResBlock3d``.
* ``resnet``: the VAE decoder's residual block (GroupNorm + swish + convolution, twice).
* ``upsample``: one octree upsampling of the VAE decoder: occupancy logits, child map,
  child features.
* ``linear`` / ``norm_linear``: the W8A8 projection of fp16 tokens, the second with the
  LayerNorm (+ modulation) in front of it.

Voxel sets are surface shells: the voxels within half a ``thickness`` of eight random
axis-aligned ellipsoids, cut to exactly ``voxels`` rows by a plane, in random row order.
A one-voxel shell has about 10 of the 27 neighbours of a voxel present, a two-voxel
shell about 18.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "hi3dv1.0-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from hi3d_amd import block as _block  # noqa: E402
from hi3d_amd import kmap, resblock, sparse, spconv, vae, w8a8  # noqa: E402
from hi3d_amd import nn as sparse_nn  # noqa: E402

EPS = 1e-6
PAIRS = {1: 10.3, 2: 17.6}
"""Present (voxel, offset) pairs per voxel of a 3x3x3 map, by shell thickness."""
COARSE = 0.3
"""Coarse voxels per fine voxel of a one-voxel shell."""
CHILDREN = 3.37
"""Children kept per parent of an upsampling."""


def _tag(i: int) -> int:
    """Keeps the streams of random numbers of one seed apart."""
    return 1_000_003 * i


# ---------------------------------------------------------------------------- cases


def listed() -> list[dict]:
    return [
        # The coarsest level of a decoder, or a small object: launches and latency.
        dict(name="layer_c128_fp16_1k5", kind="layer", voxels=1531, thickness=2, cin=128, cout=128, dtype="float16"),
        # A fine level's narrow layer in fp32 (the VAE runs in fp32 beside an fp16 transformer).
        dict(name="layer_c64_fp32_45k", kind="layer", voxels=45128, thickness=1, cin=64, cout=64, dtype="float32"),
        # An ordinary layer of a 256^3 object.
        dict(name="layer_c128_fp16_543k", kind="layer", voxels=543463, thickness=2, cin=128, cout=128, dtype="float16"),
        # The first layer of a level in bf16: its map and plan are built in the call.
        dict(name="first_c64_bf16_400k", kind="first", voxels=400003, thickness=1, cin=64, cout=64, dtype="bfloat16"),
        # Down and up one level of a 512^3 object.
        dict(name="strided_c64_c128_fp16", kind="strided", voxels=1103951, cin=64, cout=128, dtype="float16"),
        # The largest call: the residual block on a 1024^3 object.
        dict(name="block_c256_fp16_4m4", kind="block", voxels=4429513, channels=256),
        # The transformer's input/output block on a 512^3 object's coarse level, two objects in a batch.
        dict(name="resblock3d_c256_fp16", kind="resblock3d", voxels=327581, channels=256, batch=2),
        # A residual block of the VAE decoder in its default precision.
        dict(name="resnet_c128_fp32_328k", kind="resnet", voxels=327581, channels=128, dtype="float32"),
        # One octree upsampling: 328k parents to about 1.1M children.
        dict(name="upsample_c256_fp16_328k", kind="upsample", voxels=327581, channels=256, dtype="float16"),
        # The W8A8 projection at a full batch of tokens.
        dict(name="linear_65536x1024x4096", kind="linear", tokens=65536, k=1024, n=4096, rotation="h64"),
        # The transformer's MLP output on a small set of tokens.
        dict(name="linear_1030x8448x2112", kind="linear", tokens=1030, k=8448, n=2112, rotation="h64"),
        # The transformer's modulated norm and QKV projection at an ordinary, odd token count.
        dict(name="qkv_20011x2112x6336", kind="norm_linear", tokens=20011, k=2112, n=6336, modulate=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["layer", "layer", "layer", "first", "strided", "block", "resblock3d", "resnet", "upsample",
                       "linear", "linear", "norm_linear"])
    if kind in ("layer", "first"):
        dtype = rng.choice(["float16", "bfloat16", "float32"])
        cin, cout = rng.choice([(64, 64), (64, 128), (128, 128), (128, 64), (256, 128), (256, 256), (96, 160), (32, 32)])
        most = 300_000 if dtype == "float32" else 1_200_000
        return dict(kind=kind, voxels=_log_int(rng, 500, most), thickness=rng.choice([1, 2]), cin=cin, cout=cout, dtype=dtype)
    if kind == "strided":
        cin, cout = rng.choice([(64, 128), (64, 64), (128, 256)])
        return dict(kind=kind, voxels=_log_int(rng, 2000, 1_300_000), cin=cin, cout=cout,
                    dtype=rng.choice(["float16", "float16", "bfloat16", "float32"]))
    if kind == "block":
        return dict(kind=kind, voxels=_log_int(rng, 3000, 4_000_000), channels=rng.choice([128, 256]))
    if kind == "resblock3d":
        return dict(kind=kind, voxels=_log_int(rng, 3000, 2_000_000), channels=rng.choice([128, 256]), batch=rng.choice([1, 2]))
    if kind == "resnet":
        return dict(kind=kind, voxels=_log_int(rng, 2000, 330_000), channels=rng.choice([64, 128, 256]),
                    dtype=rng.choice(["float32", "float32", "float16"]))
    if kind == "upsample":
        return dict(kind=kind, voxels=_log_int(rng, 1000, 400_000), channels=rng.choice([64, 128, 256]),
                    dtype=rng.choice(["float32", "float16", "float16"]))
    k, n = rng.choice([(1024, 4096), (4096, 1024), (2112, 2112), (2112, 6336), (2112, 8448), (8448, 2112), (1024, 2112)])
    most = 65536 if k * n <= 1 << 23 else 24000
    if kind == "linear":
        return dict(kind=kind, tokens=_log_int(rng, 16, most), k=k, n=n, rotation=rng.choice(["h64", "h64", "none"]))
    if k > 4096:
        k, n = n, k
    return dict(kind=kind, tokens=_log_int(rng, 16, most), k=k, n=n, modulate=rng.random() < 0.6)


# --------------------------------------------------------------------------- inputs


def _rng(seed: int, i: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed + _tag(i))


def _normal(shape, seed: int, i: int, std: float = 1.0, mean: float = 0.0, dtype=torch.float32) -> torch.Tensor:
    x = torch.randn(shape, generator=_rng(seed, i), device="cuda", dtype=torch.float32)
    return x.mul_(std).add_(mean).to(dtype)


def shell(voxels: int, thickness: float, seed: int) -> tuple[torch.Tensor, int]:
    """``(xyz [voxels, 3] int32 in random order, grid edge)``."""
    r = np.random.default_rng(seed)
    axes, place = r.uniform(0.1, 0.4, (8, 3)), r.uniform(0.0, 1.0, (8, 3))
    centres = axes + place * (1.0 - 2.0 * axes)
    p = 1.6075  # Thomsen's approximation of an ellipsoid's area
    a, b, c = axes.T
    area = float((4 * np.pi * (((a * b) ** p + (a * c) ** p + (b * c) ** p) / 3) ** (1 / p)).sum())
    g = max(8, int(math.sqrt(1.1 * voxels / (area * thickness))) + 1)
    while True:
        keys = []
        for ax, ce in zip(axes * g, centres * g):
            lo = np.maximum(np.floor(ce - ax - thickness - 1), 0).astype(int)
            hi = np.minimum(np.ceil(ce + ax + thickness + 1), g).astype(int)
            axis = [torch.arange(int(lo[i]), int(hi[i]), device="cuda", dtype=torch.float32) + 0.5 for i in range(3)]
            q = [((v - float(ce[i])) / float(ax[i])) for i, v in enumerate(axis)]
            step = max(1, (1 << 25) // max(1, len(axis[1]) * len(axis[2])))
            for s in range(0, len(axis[0]), step):
                qx, x = q[0][s:s + step], axis[0][s:s + step]
                rr = (qx * qx)[:, None, None] + (q[1] * q[1])[None, :, None] + (q[2] * q[2])[None, None, :]
                gx, gy, gz = (v / float(ax[i]) for i, v in enumerate((qx, q[1], q[2])))
                gg = (gx * gx)[:, None, None] + (gy * gy)[None, :, None] + (gz * gz)[None, None, :]
                near = (rr.sqrt() - 1).abs() * rr.sqrt() < thickness / 2 * gg.sqrt()
                at = near.nonzero()
                key = (at[:, 0] + int(x[0].item())) * g + (at[:, 1] + int(lo[1]))
                keys.append(key * g + (at[:, 2] + int(lo[2])))
        key = torch.unique(torch.cat(keys))
        if len(key) >= voxels:
            break
        g = int(g * max(1.02, math.sqrt(1.02 * voxels / max(1, len(key))))) + 1
    key = key[:voxels][torch.randperm(voxels, generator=_rng(seed, 0), device="cuda")]
    return torch.stack([key // (g * g), key // g % g, key % g], 1).int(), g


def _rows(xyz: torch.Tensor, batch: int = 0) -> torch.Tensor:
    return torch.cat([torch.full((len(xyz), 1), batch, dtype=torch.int32, device=xyz.device), xyz], 1)


def inputs(case: dict, seed: int) -> dict:
    """Plain tensors: everything the case's values depend on."""
    kind, d = case["kind"], {}
    dt = getattr(torch, case.get("dtype", "float16"))
    if kind in ("linear", "norm_linear"):
        m, k, n = case["tokens"], case["k"], case["n"]
        x = _normal((m, k), seed, 1)
        x = torch.where(torch.rand((m, k), generator=_rng(seed, 2), device="cuda") < 0.01, 20 * x, x)
        d["x"] = x.half()
        d["w"] = _normal((n, k), seed, 3, 32.0).round_().clamp_(-127, 127).to(torch.int8)
        d["sw"] = (0.8 + 0.4 * torch.rand(n, generator=_rng(seed, 4), device="cuda")) / (32 * math.sqrt(k))
        d["bias"] = _normal((n,), seed, 5, 0.02, dtype=torch.float16)
        if kind == "norm_linear" and case["modulate"]:
            d["scale"], d["shift"] = _normal((k,), seed, 6, 0.1, 1.0, torch.float16), _normal((k,), seed, 7, 0.1, dtype=torch.float16)
        elif kind == "norm_linear":
            d["weight"], d["norm_bias"] = _normal((k,), seed, 6, 0.1, 1.0), _normal((k,), seed, 7, 0.1)
        return d
    n = case["voxels"]
    if kind == "resblock3d" and case["batch"] == 2:
        first = n // 2 + n // 16
        (xa, ga), (xb, gb) = shell(first, 1, seed), shell(n - first, 1, seed + _tag(1))
        d["indices"], d["grid"] = torch.cat([_rows(xa), _rows(xb, 1)]), max(ga, gb)
    elif kind == "strided":
        # One shell per size, turned and mirrored by the seed about an even edge, so that
        # its coarse set keeps its size.
        xyz, g = shell(n, 1, n)
        g += g % 2
        r = np.random.default_rng(seed)
        order, mirror = r.permutation(3).tolist(), torch.from_numpy(r.integers(0, 2, 3).astype(np.int32)).cuda()
        xyz = xyz[:, order][torch.randperm(n, generator=_rng(seed, 0), device="cuda")]
        d["indices"], d["grid"] = _rows(torch.where(mirror > 0, g - 1 - xyz, xyz).int().contiguous()), g
    else:
        xyz, d["grid"] = shell(n, case.get("thickness", 1), seed)
        d["indices"] = _rows(xyz)
    if kind in ("layer", "first", "strided"):
        ci, co, kv = case["cin"], case["cout"], 8 if kind == "strided" else 27
        d["x"] = _normal((n, ci), seed, 1, dtype=dt)
        d["w"] = _normal((co, kv, ci), seed, 2, 1 / math.sqrt(kv * ci), dtype=dt)
        d["b"] = _normal((co,), seed, 3, 0.02, dtype=dt)
        if kind == "strided":
            d["w_up"] = _normal((ci, 8, co), seed, 4, 1 / math.sqrt(8 * co), dtype=dt)
            d["b_up"] = _normal((ci,), seed, 5, 0.02, dtype=dt)
        return d
    c = case["channels"]
    d["x"] = _normal((n, c), seed, 1, dtype=dt)
    if kind == "block":
        d["cond"] = _normal((1024,), seed, 2)
        d["proj"], d["proj_b"] = _normal((2 * c, 1024), seed, 3, 1 / 32 / 4), _normal((2 * c,), seed, 4, 0.02)
        for i in (1, 2):
            d[f"w{i}"] = _normal((c, 27, c), seed, 4 + i, 1 / math.sqrt(27 * c), dtype=dt)
            d[f"b{i}"] = _normal((c,), seed, 6 + i, 0.02, dtype=dt)
    elif kind == "resblock3d":
        h = c // 2
        d["emb"] = _normal((case["batch"], 2112), seed, 2, dtype=dt)
        d["norm_w"], d["norm_b"] = _normal((c,), seed, 3, 0.1, 1.0, dt), _normal((c,), seed, 4, 0.1, dtype=dt)
        d["w1"], d["b1"] = _normal((h, 27, c), seed, 5, 1 / math.sqrt(27 * c), dtype=dt), _normal((h,), seed, 6, 0.02, dtype=dt)
        d["w2"], d["b2"] = _normal((h, 27, h), seed, 7, 1 / math.sqrt(27 * h), dtype=dt), _normal((h,), seed, 8, 0.02, dtype=dt)
        d["proj"], d["proj_b"] = _normal((2 * h, 2112), seed, 9, 1 / 46 / 2, dtype=dt), _normal((2 * h,), seed, 10, 0.02, dtype=dt)
        d["lin"], d["lin_b"] = _normal((c, h), seed, 11, 1 / math.sqrt(h), dtype=dt), _normal((c,), seed, 12, 0.02, dtype=dt)
    elif kind == "resnet":
        for i in (1, 2):
            d[f"gw{i}"], d[f"gb{i}"] = _normal((1, c), seed, 10 * i, 0.1, 1.0), _normal((1, c), seed, 10 * i + 1, 0.1)
            d[f"w{i}"] = _normal((27 * c, c), seed, 10 * i + 2, 1 / math.sqrt(27 * c), dtype=dt)
            d[f"b{i}"] = _normal((c,), seed, 10 * i + 3, 0.02, dtype=dt)
    else:
        d["mask"] = torch.zeros(8 * n, dtype=torch.bool, device="cuda")
        d["mask"][torch.randperm(8 * n, generator=_rng(seed, 2), device="cuda")[:int(CHILDREN * n)]] = True
        d["mask"] = d["mask"].reshape(n, 8)
        d["gw"], d["gb"] = _normal((1, c), seed, 3, 0.1, 1.0), _normal((1, c), seed, 4, 0.1)
        d["w"], d["b"] = _normal((27 * c, 8), seed, 5, 1 / math.sqrt(27 * c), dtype=dt), _normal((8,), seed, 6, 0.02, dtype=dt)
        d["proj"] = _normal((8 * c, c), seed, 7, 1 / math.sqrt(c), dtype=dt)
    return d


def _load(module, weight, bias, shape):
    with torch.no_grad():
        module.weight = torch.nn.Parameter(weight.reshape(shape))
        module.bias = torch.nn.Parameter(bias)
    return module


@torch.no_grad()
def prepare(case: dict, seed: int) -> dict:
    """What a program holds before the call: inputs, modules, and the kernel map and tile
    plan of a coordinate set that earlier layers have already used."""
    kind, d = case["kind"], inputs(case, seed)
    s = {"kind": kind, "d": d}
    if kind in ("linear", "norm_linear"):
        s["rotation"] = case.get("rotation", "h64")
        return s
    idx, g = d["indices"], d["grid"]
    if kind in ("layer", "first"):
        ci, co = case["cin"], case["cout"]
        s["conv"] = _load(spconv.SubMConv3d(ci, co, 3, indice_key="k"), d["w"], d["b"], (co, 3, 3, 3, ci))
        s["grid"] = [g, g, g]
        if kind == "layer":
            s["x"] = spconv.SparseConvTensor(d["x"], idx, s["grid"], 1)
            s["conv"](s["x"])
    elif kind == "strided":
        ci, co = case["cin"], case["cout"]
        s["down"] = _load(spconv.SparseConv3d(ci, co, 2, 2, indice_key="k"), d["w"], d["b"], (co, 2, 2, 2, ci))
        s["up"] = _load(spconv.SparseInverseConv3d(co, ci, 2, indice_key="k"), d["w_up"], d["b_up"], (ci, 2, 2, 2, co))
        s["x"] = spconv.SparseConvTensor(d["x"], idx, [g, g, g], 1)
        s["up"](s["down"](s["x"]))
    elif kind == "block":
        c = case["channels"]
        s["plan"] = kmap.build_kernel_map(idx, [g, g, g], 1).plan()
        s["weights"] = _block.ResBlockWeights(d["proj"], d["proj_b"], d["w1"].reshape(c, 3, 3, 3, c), d["b1"],
                                              d["w2"].reshape(c, 3, 3, 3, c), d["b2"])
    elif kind == "resblock3d":
        c = case["channels"]
        m = resblock.SparseResBlock3d(c, 2112).cuda().half()
        _load(m.norm1, d["norm_w"], d["norm_b"], (c,))
        _load(m.conv1.conv, d["w1"], d["b1"], (c // 2, 3, 3, 3, c))
        _load(m.conv2.conv, d["w2"], d["b2"], (c // 2, 3, 3, 3, c // 2))
        _load(m.emb_layers[1], d["proj"], d["proj_b"], (c, 2112))
        _load(m.linear, d["lin"], d["lin_b"], (c, c // 2))
        s["module"], s["x"] = m, sparse_nn.SparseTensor(d["x"], idx)
        m(s["x"], d["emb"])
    else:
        s["level"] = sparse.Level.from_coords(idx[:, 1:].contiguous())
        s["level"].plan  # built by the level's first layer
        if kind == "resnet":
            s["params"] = {"r.block.0.weights": d["gw1"], "r.block.0.bias": d["gb1"], "r.block.2.weight": d["w1"],
                           "r.block.2.bias": d["b1"], "r.block.3.weights": d["gw2"], "r.block.3.bias": d["gb2"],
                           "r.block.5.weight": d["w2"], "r.block.5.bias": d["b2"]}
        else:
            s["params"] = {"u.cls_head.fc.0.weights": d["gw"], "u.cls_head.fc.0.bias": d["gb"],
                           "u.cls_head.fc.2.weight": d["w"], "u.cls_head.fc.2.bias": d["b"], "u.proj.weight": d["proj"]}
    return s


@torch.no_grad()
def run(s: dict):
    kind, d = s["kind"], s["d"]
    if kind == "layer":
        return s["conv"](s["x"]).features
    if kind == "first":
        x = spconv.SparseConvTensor(d["x"], d["indices"], s["grid"], 1)
        y = s["conv"](x)
        return {"features": y.features, "table": x.find_indice_pair("k").kmap.table}
    if kind == "strided":
        low = s["down"](s["x"])
        return {"low": low.features, "indices": low.indices, "fine": s["up"](low).features}
    if kind == "block":
        return _block.residual_block(d["x"], s["plan"], d["cond"], s["weights"])
    if kind == "resblock3d":
        return s["module"](s["x"], d["emb"]).feats
    if kind == "resnet":
        return vae.resnet(d["x"], s["level"], s["params"], "r")
    if kind == "upsample":
        logits = vae.occupancy(d["x"], s["level"], s["params"], "u")
        y, level, _ = vae.upsample(d["x"], s["level"], s["params"], "u", mask=d["mask"])
        return {"logits": logits, "features": y, "coords": level.coords, "table": level.table}
    if kind == "linear":
        return w8a8.linear(d["x"], d["w"], d["sw"], d["bias"], rotation=s["rotation"])
    return w8a8.norm_linear(d["x"], EPS, d["w"], d["sw"], d["bias"], weight=d.get("weight"), norm_bias=d.get("norm_bias"),
                            scale=d.get("scale"), shift=d.get("shift"))


# ---------------------------------------------------------------- work and tolerance


def work(case: dict) -> dict:
    """Present pairs only; features, weights, gather tables and outputs once."""
    kind = case["kind"]
    if kind in ("linear", "norm_linear"):
        m, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": 2 * m * k + n * k + 2 * m * n + 6 * n, "flops": 2 * m * n * k}
    n, e = case["voxels"], 4 if case.get("dtype") == "float32" else 2
    pairs = PAIRS[case.get("thickness", 1)] * n
    if kind in ("layer", "first"):
        ci, co = case["cin"], case["cout"]
        table = (16 + 108) * n if kind == "first" else 108 * n
        return {"bytes": e * (n * (ci + co) + 27 * ci * co) + table, "flops": 2 * pairs * ci * co}
    if kind == "strided":
        ci, co = case["cin"], case["cout"]
        return {"bytes": 2 * e * (n * ci + COARSE * n * co + 8 * ci * co) + 10 * n, "flops": 4 * n * ci * co}
    c = case["channels"]
    if kind == "block":
        return {"bytes": e * (2 * n * c + 2 * 27 * c * c) + 108 * n, "flops": 4 * pairs * c * c}
    if kind == "resblock3d":
        h = c // 2
        return {"bytes": e * (2 * n * c + 27 * (c * h + h * h) + h * c) + 108 * n, "flops": 2 * pairs * (c * h + h * h) + 2 * n * h * c}
    if kind == "resnet":
        return {"bytes": e * (2 * n * c + 2 * 27 * c * c) + 108 * n, "flops": 4 * pairs * c * c}
    kids = int(CHILDREN * n)
    return {"bytes": e * (n * c + kids * c + 8 * c * c + 27 * 8 * c + 8 * n) + 108 * (n + kids) + 12 * (n + kids) + 8 * n,
            "flops": 2 * pairs * 8 * c + 2 * kids * c * c}


def tolerance(case: dict) -> dict:
    """About four times the error against :func:`exact` (one rounding of the output type
    after sums in fp32; the blocks round between their layers too)."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 9e-4, "max": 1e-2}
    if kind == "norm_linear":  # the codes are those of fp16 rows, whose last bit can go either way
        return {"rel": 6e-3, "max": 5e-2}
    dtype = case.get("dtype", "float16")
    if dtype == "float32":
        return {"rel": 4e-6, "max": 3e-5}
    if dtype == "bfloat16":
        return {"rel": 7e-3, "max": 4e-2}
    return {"rel": 1.1e-3, "max": 1e-2}


# ------------------------------------------------------------------------- 64 bits


def _table64(idx: torch.Tensor, g: int) -> torch.Tensor:
    """``[27, N]`` row of each neighbour in x-major offset order, -1 where absent."""
    r = idx.long()
    key = lambda b, x, y, z: ((b * (g + 2) + x + 1) * (g + 2) + y + 1) * (g + 2) + z + 1  # noqa: E731
    keys, order = torch.sort(key(*r.unbind(1)))
    out = []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                want = key(r[:, 0], r[:, 1] + dx, r[:, 2] + dy, r[:, 3] + dz)
                at = torch.searchsorted(keys, want).clamp_(max=len(keys) - 1)
                out.append(torch.where(keys[at] == want, order[at], -1))
    return torch.stack(out)


def _conv64(x, table, w, b):
    """``x [N, Cin]``, ``table [K, M]``, ``w [Cout, K, Cin]`` in float64."""
    out = torch.zeros((table.shape[1], w.shape[0]), dtype=torch.float64, device=x.device)
    if b is not None:
        out += b.double()
    for k in range(table.shape[0]):
        to = (table[k] >= 0).nonzero()[:, 0]
        if len(to):
            out.index_add_(0, to, x[table[k][to]] @ w[:, k].double().T.contiguous())
    return out


def _silu(x):
    return x * torch.sigmoid(x)


def _norm64(x, weight=None, bias=None):
    y = x - x.mean(1, keepdim=True)
    y = y / torch.sqrt((y * y).mean(1, keepdim=True) + EPS)
    return y if weight is None else y * weight.double() + bias.double()


def _gn_swish64(x, weight, bias):
    n, c = x.shape
    groups = 32 if c >= 128 else c // 4
    v = x.reshape(n, groups, c // groups)
    count = n * (c // groups) + EPS
    mean = v.sum((0, 2)) / count
    var = (v * v).sum((0, 2)) / count - mean * mean
    y = ((v - mean[None, :, None]) / torch.sqrt(var + EPS)[None, :, None]).reshape(n, c)
    return _silu(y * weight.double() + bias.double())


def _w8a8_64(v, d, rotation):
    m, k = v.shape
    if rotation == "h64":
        sign = torch.from_numpy(np.random.default_rng(314159 + k).choice([-1.0, 1.0], k)).to(v.device)
        h = torch.ones((1, 1), dtype=torch.float64, device=v.device)
        for _ in range(6):
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        v = ((v * sign).reshape(-1, 64) @ h / 8).reshape(m, k)
    s = v.abs().amax(1).clamp_min(1e-8) / 127
    q = torch.round(v / s[:, None]).clamp_(-127, 127)
    return (q @ d["w"].double().T.contiguous()) * s[:, None] * d["sw"].double() + d["bias"].double()


@torch.no_grad()
def exact(case: dict, seed: int):
    kind, d = case["kind"], inputs(case, seed)
    x = d["x"].double()
    if kind == "linear":
        return _w8a8_64(x, d, case["rotation"])
    if kind == "norm_linear":
        y = _norm64(x, d.get("weight"), d.get("norm_bias"))
        if "scale" in d:
            y = y * d["scale"].double() + d["shift"].double()
        return _w8a8_64(y, d, "h64")
    if kind == "strided":
        idx, g = d["indices"].long(), d["grid"]
        half = idx.clone()
        half[:, 1:] //= 2
        e = g // 2 + 1
        key = ((half[:, 0] * e + half[:, 1]) * e + half[:, 2]) * e + half[:, 3]
        uniq, parent = torch.unique(key, return_inverse=True)
        slot = (idx[:, 1] & 1) * 4 + (idx[:, 2] & 1) * 2 + (idx[:, 3] & 1)
        down = torch.full((8, len(uniq)), -1, dtype=torch.long, device=idx.device)
        down[slot, parent] = torch.arange(len(idx), device=idx.device)
        low = _conv64(x, down, d["w"], d["b"])
        up = torch.stack([torch.where(slot == k, parent, -1) for k in range(8)])
        return {"low": low, "indices": None, "fine": _conv64(low, up, d["w_up"], d["b_up"])}
    table = _table64(d["indices"], d["grid"])
    if kind == "layer":
        return _conv64(x, table, d["w"], d["b"])
    if kind == "first":
        return {"features": _conv64(x, table, d["w"], d["b"]), "table": None}
    if kind == "block":
        scale, shift = (d["proj"].double() @ d["cond"].double() + d["proj_b"].double()).chunk(2)
        h = _silu(_conv64(_norm64(x) * (1 + scale) + shift, table, d["w1"], d["b1"]))
        return _conv64(h, table, d["w2"], d["b2"]) + x
    if kind == "resblock3d":
        batch = d["indices"][:, 0].long()
        mod = _silu(d["emb"].double()) @ d["proj"].double().T.contiguous() + d["proj_b"].double()
        scale, shift = mod[batch].chunk(2, 1)
        h = _conv64(_silu(_norm64(x, d["norm_w"], d["norm_b"])), table, d["w1"], d["b1"])
        h = _silu(_conv64(_silu(_norm64(h) * (1 + scale) + shift), table, d["w2"], d["b2"]))
        return h @ d["lin"].double().T.contiguous() + d["lin_b"].double() + x
    spconv_layout = lambda w: w.T.reshape(w.shape[1], 27, -1)  # noqa: E731
    if kind == "resnet":
        h = x
        for i in (1, 2):
            h = _conv64(_gn_swish64(h, d[f"gw{i}"], d[f"gb{i}"]), table, spconv_layout(d[f"w{i}"]), d[f"b{i}"])
        return h + x
    logits = _conv64(_gn_swish64(x, d["gw"], d["gb"]), table, spconv_layout(d["w"]), d["b"])
    parent, slot = d["mask"].nonzero().unbind(1)
    c = x.shape[1]
    feats = torch.empty((len(parent), c), dtype=torch.float64, device=x.device)
    for k in range(8):
        to = (slot == k).nonzero()[:, 0]
        feats[to] = x[parent[to]] @ d["proj"][k * c:(k + 1) * c].double().T.contiguous()
    return {"logits": logits, "features": feats, "coords": None, "table": None}
