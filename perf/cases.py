"""Performance cases: the calls a program makes on this framework, over the
sizes, widths, dtypes and dataflows it makes them with.

Four kinds of case:

* ``map``   -- one kernel map, ``F.build_kmap`` on sorted packed keys;
* ``maps``  -- what a network needs before its first layer: ``order()`` of raw
  voxels and features, then ``KernelMapCache.add_all_kernel_maps``;
* ``layer`` -- one ``SparseConv`` call on maps that are in the cache (every
  dataflow, fp16 and fp32, submanifold, strided and transposed), or one fused
  residual block;
* ``net``   -- a whole inference step on a new scene: ``order()``, the
  network-wide map build and the forward pass.

A module documents its dataflow numbering in ``spira_amd.nn.conv``; 2 is what a
``SparseConv`` is constructed with, 0 is what the end-to-end networks run.
"""
from __future__ import annotations

import functools
import math
from typing import Dict, List, Tuple

import numpy as np
import torch

import spira_amd
from spira_amd import nn as spnn
from spira_amd import scenes
from spira_amd.networks import SparseResBlock, SparseResNetLarge, SparseResUNet42, kmap_schedule
from spira_amd.nn import functional as F

_SCENES = {"objects": scenes.spheres_planes, "lidar": scenes.lidar, "indoor": scenes.indoor,
           "blobs": scenes.lidar_blobs}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _map(name, scene, n, k, stride, dataflow, double):
    return {"name": name, "kind": "map", "scene": scene, "n": n, "k": k, "stride": stride, "dataflow": dataflow,
            "double": double}


def _layer(name, scene, n, k, cin, cout, dataflow, dtype, form="same"):
    return {"name": name, "kind": "layer", "scene": scene, "n": n, "k": k, "cin": cin, "cout": cout,
            "dataflow": dataflow, "dtype": dtype, "form": form}


def listed() -> List[dict]:
    return [
        # a small object scan with 32-bit keys: the smallest map, where launches and latency count
        _map("map_objects_20k_k3", "objects", 20_000, 3, 1, 0, False),
        # the large search: one LiDAR sweep, 125 offsets, 64-bit keys
        _map("map_lidar_100k_k5", "lidar", 100_000, 5, 1, 0, True),
        # the map of a layer as constructed (masks for gather / GEMM / scatter)
        _map("map_lidar_100k_k3_masks", "lidar", 100_000, 3, 1, 2, True),
        # a room scan's maps for a whole UNet: sort, four downsampled levels, nine maps
        {"name": "maps_indoor_200k", "kind": "maps", "scene": "indoor", "n": 200_000, "net": "UNet", "cin": 3},
        # one output-stationary layer on a LiDAR sweep, the middle of the width sweep
        _layer("os_f16_lidar_100k_c64", "lidar", 100_000, 3, 64, 64, 0, "f16"),
        # the same dataflow in fp32 on a small scan (a network kept in full precision)
        _layer("os_f32_objects_20k_c32", "objects", 20_000, 3, 32, 32, 0, "f32"),
        # the fused weight-stationary dataflow, which the selector may pick per layer
        _layer("ws_f16_indoor_100k_c64", "indoor", 100_000, 3, 64, 64, 1, "f16"),
        # a layer exactly as constructed: fp32, gather / GEMM / scatter
        _layer("gs_f32_objects_20k_c32", "objects", 20_000, 3, 32, 64, 2, "f32"),
        # a hybrid layer: the dense offsets output-stationary, the others gather / GEMM / scatter
        _layer("hs_f16_lidar_100k_c64", "lidar", 100_000, 3, 64, 64, 6, "f16"),
        # the decoder's full-resolution residual block after a skip concatenation, fused for inference
        _layer("block_f16_indoor_200k_c96", "indoor", 200_000, 3, 128, 96, 0, "f16", form="block"),
        # a small scene through the k = 5 residual network
        {"name": "net_blobs_30k_resnet_large", "kind": "net", "scene": "blobs", "n": 30_000, "net": "ResNetLarge",
         "cin": 4},
        # a room scan through the 42-layer UNet: the headline step
        {"name": "net_indoor_200k_unet42", "kind": "net", "scene": "indoor", "n": 200_000, "net": "UNet", "cin": 3},
    ]


def draw(rng) -> dict:
    scene = rng.choice(["objects", "lidar", "indoor"])

    def size(lo, hi):
        if scene == "objects":  # (what its surfaces hold)
            hi = min(hi, 60_000)
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    u = rng.random()
    if u < 0.25:
        k = rng.choice([3, 3, 5])
        stride = rng.choice([1, 1, 2])
        # (hybrid maps are built for submanifold layers)
        dataflow = rng.choice([0, 0, 1, 2] + ([3, 4, 5, 6] if stride == 1 else []))
        if stride == 2 and dataflow == 1:
            k = 2  # (the UNet's down-sampling maps)
        return _map("", scene, size(4_000, 200_000 if k < 5 else 100_000), k, stride, dataflow,
                    rng.random() < 0.7) | {"name": None}
    if u < 0.35:
        return {"kind": "maps", "scene": scene, "n": size(5_000, 200_000), "net": rng.choice(["UNet", "ResNetLarge"]),
                "cin": rng.choice([3, 4]), "name": None}
    if u < 0.90:
        form = rng.choice(["same"] * 5 + ["down", "up", "block"])
        dtype = rng.choice(["f16", "f16", "f32"])
        k = 2 if form in ("down", "up") else rng.choice([3, 3, 3, 5])
        widths = [16, 20, 24, 32, 48, 64, 96, 128] + ([256] if dtype == "f16" and k != 5 else [])
        cin, cout = rng.choice([3, 4] + widths), rng.choice(widths)
        hybrid = [3, 4, 5, 6] if form == "same" else []
        dataflow = 0 if form == "block" else rng.choice([0, 0, 0, 1, 1, 2, 2] + hybrid)
        if form == "block":
            dtype, k, cin = "f16", 3, rng.choice(widths)
        hi = (200_000 if dtype == "f16" else 60_000) if k != 5 else 40_000
        return _layer("", scene, size(3_000, hi), k, cin, cout, dataflow, dtype, form) | {"name": None}
    return {"kind": "net", "scene": scene, "n": size(5_000, 120_000), "net": rng.choice(["UNet", "ResNetLarge"]),
            "cin": rng.choice([3, 4]), "name": None}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device() -> torch.device:
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=_device()).manual_seed(1_000_003 * seed + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=_device())


@functools.lru_cache(maxsize=64)
def _scene(scene: str, n: int) -> np.ndarray:
    return _SCENES[scene](n)


def _voxels(case: dict, seed: int) -> torch.Tensor:
    """The case's scene as another scan would see it: mirrored, turned, moved
    by whole 16-voxel cells and shuffled by the seed (so that every seed has
    the same number of voxels on every level), away from the origin."""
    rng = np.random.default_rng(1000 + seed)
    v = _scene(case["scene"], case["n"])
    size = (v.max(axis=0) // 16 + 1) * 16
    flip = rng.random(3) < 0.5
    v = np.where(flip, size - 1 - v, v) + 16 * rng.integers(1, 4, 3)
    if rng.random() < 0.5:
        v = v[:, [1, 0, 2]]
    v = np.ascontiguousarray(v[rng.permutation(len(v))].astype(np.int32))
    return torch.from_numpy(v).to(_device())


def _dtype(case: dict) -> torch.dtype:
    return torch.float32 if case.get("dtype") == "f32" else torch.float16


def _norm(g, sd: dict, prefix: str, c: int) -> None:
    """Batch-norm statistics and affine parameters of a trained network's size
    (with the defaults a random network shrinks its activations to nothing)."""
    sd[prefix + ".running_mean"] = 0.1 * _randn(g, c)
    sd[prefix + ".running_var"] = 0.5 + torch.rand(c, generator=g, device=_device())
    sd[prefix + ".weight"] = 0.5 + torch.rand(c, generator=g, device=_device())
    sd[prefix + ".bias"] = 0.1 * _randn(g, c)


def _kernel(g, volume: int, cin: int, cout: int) -> torch.Tensor:
    # (a quarter of the offsets have a neighbour: activations of order one through the residual sums)
    return _randn(g, volume, cin, cout) * math.sqrt(0.5 / (cin * max(1.0, volume / 4)))


def _conv_bn(g, sd, conv, bn, volume, cin, cout):
    sd[conv + ".kernel"] = _kernel(g, volume, cin, cout)
    _norm(g, sd, bn, cout)


def _block(g, sd, p, cin, cout, volume):
    _conv_bn(g, sd, p + "main.0", p + "main.1", volume, cin, cout)
    _conv_bn(g, sd, p + "main.3", p + "main.4", volume, cout, cout)
    if cin != cout:
        _conv_bn(g, sd, p + "shortcut.0", p + "shortcut.1", 1, cin, cout)


_UNET = [32, 32, 64, 128, 256, 256, 128, 96, 96]
_RESNET_LARGE = [(16, 1), (32, 2), (64, 2), (128, 2)]


def _weights(net: str, cin: int, seed: int) -> Dict[str, torch.Tensor]:
    """Seeded fp16 parameters of a network, under its state_dict names."""
    g, sd = _gen(seed), {}
    if net == "UNet":
        ch = _UNET
        _conv_bn(g, sd, "stem.0", "stem.1", 27, cin, ch[0])
        _conv_bn(g, sd, "stem.3", "stem.4", 27, ch[0], ch[0])
        for k in range(4):
            _conv_bn(g, sd, f"encoders.{k}.0.0", f"encoders.{k}.0.1", 8, ch[k], ch[k])
            _block(g, sd, f"encoders.{k}.1.", ch[k], ch[k + 1], 27)
            _block(g, sd, f"encoders.{k}.2.", ch[k + 1], ch[k + 1], 27)
            p = f"decoders.{k}."
            _conv_bn(g, sd, p + "upsample.0", p + "upsample.1", 8, ch[k + 4], ch[k + 5])
            _block(g, sd, p + "fuse.0.", ch[k + 5] + ch[3 - k], ch[k + 5], 27)
            _block(g, sd, p + "fuse.1.", ch[k + 5], ch[k + 5], 27)
    else:
        for i, (c, _) in enumerate(_RESNET_LARGE):
            _conv_bn(g, sd, f"{i}.0.0", f"{i}.0.1", 125, cin, c)
            _block(g, sd, f"{i}.1.", c, c, 125)
            _block(g, sd, f"{i}.2.", c, c, 125)
            cin = c
    return {k: v.half() for k, v in sd.items()}


def _load(model: torch.nn.Module, sd: Dict[str, torch.Tensor]) -> torch.nn.Module:
    model = model.to(_device()).half().eval()
    missing, unexpected = model.load_state_dict(sd, strict=False)
    if unexpected or any(not m.endswith("num_batches_tracked") for m in missing):
        raise RuntimeError(f"state_dict mismatch: {missing} {unexpected}")
    for m in model.modules():
        if isinstance(m, spnn.SparseConv):
            m.tunable_config["map_dataflow"] = 0
    return spnn.fuse_epilogues(model)


def _layer_inputs(case: dict, seed: int):
    """(voxels, input features, weights): features row i belong to sorted key
    i of the layer's input level; weights are a tensor or (block) a dict."""
    g = _gen(seed)
    dt = _dtype(case)
    vox = _voxels(case, seed)
    rows = int(_down(_key(vox), 2).numel()) if case["form"] == "up" else vox.shape[0]
    x = _randn(g, rows, case["cin"]).to(dt)
    if case["form"] == "block":
        w = {}
        _block(g, w, "", case["cin"], case["cout"], case["k"] ** 3)
        w = {k: v.to(dt) for k, v in w.items()}
    else:
        w = _kernel(g, case["k"] ** 3, case["cin"], case["cout"]).to(dt)
    return vox, x, w


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "map":
        keys, _ = F.flat_sort(_voxels(case, seed), case["double"])
        s = case["stride"]
        targets = keys if s == 1 else F.downsample(keys, (s, s, s))
        return {"case": case, "sources": keys, "targets": targets}
    if kind in ("maps", "net"):
        vox = _voxels(case, seed)
        state = {"case": case, "voxels": vox, "features": _randn(_gen(seed + 1), vox.shape[0], case["cin"]).half(),
                 "schedule": kmap_schedule(case["net"]), "cache": spnn.KernelMapCache()}
        if kind == "net":
            model = (SparseResUNet42 if case["net"] == "UNet" else SparseResNetLarge)(in_channels=case["cin"])
            state["model"] = _load(model, _weights(case["net"], case["cin"], seed))
            spira_amd.set_kernel_map_cache(state["model"], state["cache"])
        return state
    vox, x, w = _layer_inputs(case, seed)
    keys, _ = F.flat_sort(vox, True)
    k, d, form = case["k"], case["dataflow"], case["form"]
    cache = spnn.KernelMapCache()
    one, two = (1, 1, 1), (2, 2, 2)
    if form in ("same", "block"):
        module = (SparseResBlock(case["cin"], case["cout"], k) if form == "block"
                  else spnn.SparseConv(case["cin"], case["cout"], k))
        cache.add_all_kernel_maps(keys, [k], [one, one], [], one, [d])
        inp = spira_amd.SparseTensor(keys, x, stride=1)
    else:
        module = spnn.SparseConv(case["cin"], case["cout"], k, stride=2, transposed=form == "up")
        cache.add_all_kernel_maps(keys, [3, k], [one, one, two], [two], one, [0, d])
        coarse = cache.get_target_coordinates(keys, one, two)
        inp = spira_amd.SparseTensor(coarse, x, stride=2) if form == "up" else spira_amd.SparseTensor(keys, x, stride=1)
    if form == "block":
        module = _load(module, w)
    else:
        module = module.to(device=_device(), dtype=_dtype(case)).eval()
        module.load_state_dict({"kernel": w})
        module.tunable_config["map_dataflow"] = d
    spira_amd.set_kernel_map_cache(module, cache)
    return {"case": case, "module": module, "input": inp, "cache": cache}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state: dict):
    case = state["case"]
    with torch.no_grad():
        if case["kind"] == "map":
            m = F.build_kmap(state["sources"], state["targets"], case["k"], 1, case["dataflow"])
            return [t for t in m[2:] if isinstance(t, torch.Tensor)]
        if case["kind"] == "layer":
            return state["module"](state["input"]).features
        cache = state["cache"]
        cache.reset()
        x = spira_amd.SparseTensor(coordinates=state["voxels"], features=state["features"], double=True)
        x.order()
        ts, ks, ss = state["schedule"]
        cache.add_all_kernel_maps(x.coordinates, ks, ss, ts, (1, 1, 1), [0] * len(ks))
        if case["kind"] == "net":
            return [y.features for y in state["model"](x)]
        out = [x.coordinates, x.features]
        stride = (1, 1, 1)
        for i, k in enumerate(ks):
            target = tuple(ss[i + 1])
            coords = cache.get_target_coordinates(x.coordinates, stride, target)
            out += [coords, cache.get_kernel_map(x.coordinates, stride, coords, target, k, 0)[2]]
            stride = target
        return out


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _key(vox: torch.Tensor) -> torch.Tensor:
    v = vox.to(torch.int64)
    return (v[:, 0] << 40) + (v[:, 1] << 16) + v[:, 2]


def _down(keys: torch.Tensor, s: int) -> torch.Tensor:
    x, y, z = keys >> 40, (keys >> 16) & 0xFFFFFF, keys & 0xFFFF
    return torch.unique((x // s * s << 40) + (y // s * s << 16) + z // s * s)


def _offsets(k: int) -> List[int]:
    lo = -(k // 2) if k % 2 else -(k // 2) + 1
    return list(range(lo, lo + k))


def _neighbours(src: torch.Tensor, tgt: torch.Tensor, k: int, s: int) -> List[torch.Tensor]:
    """Per offset (x-major, z innermost) the source index of every target, or -1."""
    out = []
    for dx in _offsets(k):
        for dy in _offsets(k):
            for dz in _offsets(k):
                q = tgt + ((s * dx << 40) + (s * dy << 16) + s * dz)
                at = torch.searchsorted(src, q).clamp(max=src.numel() - 1)
                out.append(torch.where(src[at] == q, at, -1))
    return out


def _apply(nb: List[torch.Tensor], x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    y = torch.zeros(nb[0].numel(), w.shape[2], dtype=x.dtype, device=x.device)
    for j, idx in enumerate(nb):
        t = torch.nonzero(idx >= 0).flatten()
        if t.numel():
            y.index_add_(0, t, x[idx[t]] @ w[j])
    return y


def _apply_transposed(nb, x, w, rows):
    """Targets of a transposed layer are the sources of the forward map."""
    y = torch.zeros(rows, w.shape[2], dtype=x.dtype, device=x.device)
    for j, idx in enumerate(nb):
        t = torch.nonzero(idx >= 0).flatten()
        if t.numel():
            y.index_add_(0, idx[t], x[t] @ w[j])
    return y


def _row_order(k: int, dataflow: int) -> List[int]:
    """Weight row j of a dataflow holds offset _row_order(...)[j] of the
    x-major list: z-major for 0, x-major for 1 and 2, the offsets nearest the
    centre first for the hybrids."""
    if dataflow == 0:
        return [o * k + z for z in range(k) for o in range(k * k)]
    if dataflow <= 2:
        return list(range(k ** 3))
    l1 = [abs(a) + abs(b) + abs(c) for a in _offsets(k) for b in _offsets(k) for c in _offsets(k)]
    near = (dataflow - 1) // 2
    return [i for i, v in enumerate(l1) if v < near] + [i for i, v in enumerate(l1) if v >= near]


def _bn(x, sd, p, eps=1e-5):
    v = {n: sd[f"{p}.{n}"].double() for n in ("running_mean", "running_var", "weight", "bias")}
    return (x - v["running_mean"]) / torch.sqrt(v["running_var"] + eps) * v["weight"] + v["bias"]


class _Exact:
    """A network's layers in 64 bits on one scene."""

    def __init__(self, keys, sd):
        self.levels, self.maps, self.sd = {1: keys}, {}, sd

    def nb(self, src, tgt, k):
        key = (src, tgt, k)
        if key not in self.maps:
            for s in (src, tgt):
                if s not in self.levels:
                    self.levels[s] = _down(self.levels[1], s)
            nb = _neighbours(self.levels[src], self.levels[tgt], k, src)
            self.maps[key] = [nb[i] for i in _row_order(k, 0)]
        return self.maps[key]

    def conv_bn(self, x, conv, bn, src, tgt, k):
        w = self.sd[conv + ".kernel"].double()
        if k == 1:
            y = x @ w[0]
        elif tgt >= src:
            y = _apply(self.nb(src, tgt, k), x, w)
        else:
            y = _apply_transposed(self.nb(tgt, src, k), x, w, self.levels[tgt].numel())
        return _bn(y, self.sd, bn)

    def block(self, x, p, s, k):
        h = self.conv_bn(x, p + "main.0", p + "main.1", s, s, k).relu()
        h = self.conv_bn(h, p + "main.3", p + "main.4", s, s, k)
        if p + "shortcut.0.kernel" in self.sd:
            x = self.conv_bn(x, p + "shortcut.0", p + "shortcut.1", s, s, 1)
        return (h + x).relu()

    def unet(self, x):
        x = self.conv_bn(x, "stem.0", "stem.1", 1, 1, 3).relu()
        x = self.conv_bn(x, "stem.3", "stem.4", 1, 1, 3).relu()
        skips = [x]
        for k in range(4):
            s = 2 ** k
            x = self.conv_bn(x, f"encoders.{k}.0.0", f"encoders.{k}.0.1", s, 2 * s, 2).relu()
            x = self.block(x, f"encoders.{k}.1.", 2 * s, 3)
            x = self.block(x, f"encoders.{k}.2.", 2 * s, 3)
            skips.append(x)
        outs = list(skips)
        for k in range(4):
            s, p = 2 ** (3 - k), f"decoders.{k}."
            x = self.conv_bn(x, p + "upsample.0", p + "upsample.1", 2 * s, s, 2).relu()
            x = self.block(torch.cat([x, skips[3 - k]], 1), p + "fuse.0.", s, 3)
            x = self.block(x, p + "fuse.1.", s, 3)
            outs.append(x)
        return outs

    def resnet_large(self, x):
        outs, s = [], 1
        for i, (_, step) in enumerate(_RESNET_LARGE):
            x = self.conv_bn(x, f"{i}.0.0", f"{i}.0.1", s, s * step, 5).relu()
            s *= step
            x = self.block(self.block(x, f"{i}.1.", s, 5), f"{i}.2.", s, 5)
            outs.append(x)
        return outs


def exact(case: dict, seed: int):
    if case["kind"] == "layer":
        vox, x, w = _layer_inputs(case, seed)
        keys = torch.sort(_key(vox)).values
        x = x.double()
        if case["form"] == "block":
            return _Exact(keys, w).block(x, "", 1, case["k"])
        k, d = case["k"], case["dataflow"]
        coarse = keys if case["form"] == "same" else _down(keys, 2)
        nb = _neighbours(keys, coarse, k, 1)
        nb = [nb[i] for i in _row_order(k, d)]
        w = w.double()
        if case["form"] == "up":
            return _apply_transposed(nb, x, w, keys.numel())
        return _apply(nb, x, w)
    if case["kind"] == "net":
        vox = _voxels(case, seed)
        keys, perm = torch.sort(_key(vox))
        x = _randn(_gen(seed + 1), vox.shape[0], case["cin"]).half()[perm].double()
        ex = _Exact(keys, _weights(case["net"], case["cin"], seed))
        return ex.unet(x) if case["net"] == "UNet" else ex.resnet_large(x)
    return None  # (keys, indices and permuted inputs: compared bit for bit)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _levels(scene: str, n: int) -> Tuple[torch.Tensor, ...]:
    keys = torch.sort(_key(_voxels({"scene": scene, "n": n}, 0))).values
    return (keys,) + tuple(_down(keys, s) for s in (2, 4, 8, 16))


@functools.lru_cache(maxsize=256)
def _geometry(scene: str, n: int, src: int, tgt: int, k: int) -> Tuple[int, int, int]:
    """(sources, targets, valid pairs) of a scene's map from level src to tgt."""
    lv = _levels(scene, n)
    a, b = lv[int(math.log2(src))], lv[int(math.log2(tgt))]
    pairs = sum(int((i >= 0).sum()) for i in _neighbours(a, b, k, src))
    return a.numel(), b.numel(), pairs


def _conv_work(g, k, cin, cout, size):
    s, t, p = g
    return {"bytes": size * (s * cin + t * cout) + size * k ** 3 * cin * cout + 4 * k ** 3 * t,
            "flops": 2 * p * cin * cout}


def _sum(parts):
    return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}


def _dense_work(n, cin, cout):
    return {"bytes": 2 * n * (cin + cout) + 2 * cin * cout, "flops": 2 * n * cin * cout}


def _block_work(geo, k, cin, cout):
    parts = [_conv_work(geo, k, cin, cout, 2), _conv_work(geo, k, cout, cout, 2)]
    if cin != cout:
        parts.append(_dense_work(geo[1], cin, cout))
    return _sum(parts)


def _maps_work(case):
    n, cin = case["n"], case["cin"]
    _, ks, ss = kmap_schedule(case["net"])
    total = _levels(case["scene"], n)[0].numel() * (12 + 8 + 4 * cin)  # voxels in, keys out, features in and out
    for i, k in enumerate(ks):
        s, t, _ = _geometry(case["scene"], n, ss[i][0], ss[i + 1][0], k[0])
        total += 8 * s + 8 * t + 4 * k[0] ** 3 * t
    return {"bytes": total, "flops": 0}


def work(case: dict) -> dict:
    scene, n = case["scene"], case["n"]
    if case["kind"] == "map":
        s, t, p = _geometry(scene, n, 1, case["stride"], case["k"])
        key, volume, d = (8 if case["double"] else 4), case["k"] ** 3, case["dataflow"]
        total = key * (s + t) + 4 * volume * t
        if d % 2 == 1:
            total += 4 * p  # (pairs of half the offsets, two words each)
        elif d > 0:
            total += 4 * volume * (s + t)
        return {"bytes": total, "flops": 0}
    if case["kind"] == "maps":
        return _maps_work(case)
    if case["kind"] == "layer":
        cin, cout, k, size = case["cin"], case["cout"], case["k"], 4 if case["dtype"] == "f32" else 2
        if case["form"] == "block":
            return _block_work(_geometry(scene, n, 1, 1, k), k, cin, cout)
        geo = _geometry(scene, n, 1, 1 if case["form"] == "same" else 2, k)
        if case["form"] == "up":
            geo = (geo[1], geo[0], geo[2])
        return _conv_work(geo, k, cin, cout, size)
    parts = [_maps_work(case)]
    cin = case["cin"]

    def conv(src, tgt, k, a, b):
        geo = _geometry(scene, n, min(src, tgt), max(src, tgt), k)
        parts.append(_conv_work(geo if src <= tgt else (geo[1], geo[0], geo[2]), k, a, b, 2))

    if case["net"] == "UNet":
        ch = _UNET
        conv(1, 1, 3, cin, ch[0])
        conv(1, 1, 3, ch[0], ch[0])
        for k in range(4):
            s, u = 2 ** k, 2 ** (3 - k)
            conv(s, 2 * s, 2, ch[k], ch[k])
            parts.append(_block_work(_geometry(scene, n, 2 * s, 2 * s, 3), 3, ch[k], ch[k + 1]))
            parts.append(_block_work(_geometry(scene, n, 2 * s, 2 * s, 3), 3, ch[k + 1], ch[k + 1]))
            conv(2 * u, u, 2, ch[k + 4], ch[k + 5])
            parts.append(_block_work(_geometry(scene, n, u, u, 3), 3, ch[k + 5] + ch[3 - k], ch[k + 5]))
            parts.append(_block_work(_geometry(scene, n, u, u, 3), 3, ch[k + 5], ch[k + 5]))
    else:
        s = 1
        for c, step in _RESNET_LARGE:
            conv(s, s * step, 5, cin, c)
            s *= step
            parts += [_block_work(_geometry(scene, n, s, s, 5), 5, c, c)] * 2
            cin = c
    return _sum(parts)


def tolerance(case: dict):
    if case["kind"] in ("map", "maps"):
        return "exact"
    if case["kind"] == "net":
        # (fp16 activations rounded again after each of 20 to 42 layers)
        return {"rel": 2.5e-3}
    if case["dtype"] == "f32":
        return {"rel": 1e-6}
    # fp16 outputs of fp32 sums; a block rounds its activations once more
    return {"rel": 1.2e-3 if case["form"] == "block" else 8e-4}
