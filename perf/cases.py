"""Representative work of the sparse-voxel library, as callables.

Each case is a dict of plain values.  `prepare` makes what a caller holds
before the call (coordinates, features, weights and kept grids on the GPU),
`run` is one pass through the public entry points of the Python binding,
`work` the bytes and flops the pass cannot do without, `exact` the same
outputs in 64 bits from plain torch, and `tolerance` the difference that
rounding alone explains.

Voxel sets are shells of random axis-aligned ellipsoids (a surface, two voxels
thick), rows sorted by (batch, x, y, z).  A case's `geometry` fixes the
ellipsoids; the seed turns the grid by one of the 48 symmetries of the cube, so
other seeds are other coordinates with the same number of voxels and of
neighbour pairs, and draws the features and weights.
"""

from __future__ import annotations

import math
import random
import sys
from functools import lru_cache
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "pixal3d.cpp_amd" / "python"))

import pxs as P  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
CODES = {"f32": P.PXS_F32, "bf16": P.PXS_BF16}
SIZE = {"f32": 4, "bf16": 2}


# ---- cases -----------------------------------------------------------------

def listed():
    return [
        # A single small submanifold convolution of unknown extents, as a
        # caller of the drop-in makes it: hash, neighbour map, 32 -> 48.
        dict(name="conv_small_f32", kind="conv", dtype="f32", lookup="hash", grid=16,
             shells="4-7;3-6", geometry=7, cin=32, cout=48),
        # One fp32 submanifold convolution over a 64^3 grid, 16k voxels.
        dict(name="conv_64_f32", kind="conv", dtype="f32", lookup="grid", grid=64,
             shells="16-30", geometry=4, cin=64, cout=64),
        # A level of a sparse U-Net encoder, topology included: the grid
        # insert, SubMConv3d, stride-2 convolution, SubMConv3d on the coarse
        # level (162k voxels, batch 2 of different lengths).
        dict(name="unet_128", kind="unet", grid=128, shells="22-36,18-30,26-40;26-44,22-38,30-50",
             geometry=2, c1=128, c2=256),
        # A decoder's wide convolution and subdivision: SubMConv3d 768 -> 8 x 192
        # over a 64^3 grid, every row split into its 8 children.
        dict(name="upsample_64", kind="upsample", grid=64, shells="20-30,14-26", geometry=4,
             cin=768, out=192),
        # The first up-block of the shape decoder, predicting which children
        # exist (those the refined surface meets): 10k rows, 1024 -> 512.
        dict(name="c2s_pred_64", kind="c2s", dtype="bf16", grid=64, shells="18-22", geometry=7,
             channels=1024, out=512),
        # The whole texture decoder, guided by the shape's subdivisions:
        # 64^3 latents to the 1024^3 surface, five levels of 1024..64 channels.
        dict(name="decoder_64", kind="decoder", dtype="bf16", grid=64, shells="18-22", geometry=7,
             channels="1024,512,256,128,64", latent=32, out=6),
        # Full self-attention over a ragged batch: QKV, per-head RMS norm,
        # attention, output projection.
        dict(name="attn_32k", kind="attn", dtype="bf16", lengths="12288,20480", heads=16,
             head_dim=64),
        # Two shifted-window attention layers with their partitions.
        dict(name="swin_64", kind="swin", grid=64, shells="20-30,14-26", geometry=4, window=8,
             heads=12),
        # One block of the large flow model at its largest voxel count.
        dict(name="block_42k", kind="block", dtype="bf16", grid=64, shells="24-31,18-30,12-24",
             geometry=5, width=1024, mlp=4096, tokens=1370),
        # The same block in 32 bits on a small object, as the drop-in calls it.
        dict(name="block_4k_f32", kind="block", dtype="f32", grid=32, shells="11-15", geometry=3,
             width=1024, mlp=4096, tokens=1370),
        # A whole flow forward (24 blocks) on a small object: launches and
        # weight traffic count as much as the arithmetic.
        dict(name="flow_1k", kind="flow", dtype="bf16", grid=32, shells="5-9", geometry=5,
             width=1024, mlp=4096, blocks=24, tokens=1370),
        # The decoder's fp32 linear at the rows of its third level.
        dict(name="linear_207k_f32", kind="linear", dtype="f32", rows=206980, cin=1024, cout=256),
    ]


def draw(rng: random.Random):
    """One more case of the listed kinds, over the whole range of sizes."""

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def shells(grid, items=1, lo=0.25, hi=0.46):
        out = []
        for _ in range(items):
            parts = []
            for _ in range(rng.randint(1, 2)):
                a = rng.uniform(lo, hi - 0.04) * grid
                parts.append(f"{a:.2f}-{rng.uniform(a + 0.02 * grid, hi * grid):.2f}")
            out.append(",".join(parts))
        return ";".join(out)

    geo = rng.randrange(1 << 20)
    kind = rng.choice(["conv", "conv", "unet", "upsample", "c2s", "decoder", "attn", "swin",
                       "block", "flow", "linear"])
    if kind == "conv":
        grid = rng.choice([14, 16, 24, 32, 45, 48, 64, 90, 128])
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]),
                    lookup=rng.choice(["grid", "hash", "bricks"]), grid=grid,
                    shells=shells(grid, rng.randint(1, 2)), geometry=geo,
                    cin=rng.choice([16, 32, 40, 64, 96, 128]),
                    cout=rng.choice([16, 36, 48, 64, 72, 128, 192]))
    if kind == "unet":
        grid = rng.choice([16, 32, 50, 64, 96, 128])
        c1 = rng.choice([64, 128])
        return dict(kind=kind, grid=grid, shells=shells(grid, rng.randint(1, 2)), geometry=geo,
                    c1=c1, c2=rng.choice([c1, 2 * c1]))
    if kind == "upsample":
        grid = rng.choice([16, 24, 32, 48, 64])
        return dict(kind=kind, grid=grid, shells=shells(grid), geometry=geo,
                    cin=rng.choice([128, 256, 384, 768]), out=rng.choice([64, 96, 192]))
    if kind == "c2s":
        grid = rng.choice([16, 24, 32, 48, 64])
        channels = rng.choice([128, 256, 512, 1024])
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16", "bf16"]) if channels < 512 else "bf16",
                    grid=grid, shells=shells(grid, 1, 0.2, 0.35), geometry=geo, channels=channels,
                    out=channels // 2)
    if kind == "decoder":
        grid = rng.choice([16, 24, 32, 64])
        levels = rng.randint(2, 4)
        return dict(kind=kind, dtype="bf16", grid=grid, shells=shells(grid, 1, 0.2, 0.33),
                    geometry=geo, channels=",".join(str(512 >> i) for i in range(levels)),
                    latent=32, out=rng.choice([6, 7]))
    if kind == "attn":
        items = rng.randint(1, 4)
        lengths = [log(48, 20000 if items < 3 else 8000) for _ in range(items)]
        f32 = max(lengths) < 6000 and rng.random() < 0.4
        return dict(kind=kind, dtype="f32" if f32 else "bf16",
                    lengths=",".join(str(n) for n in lengths), heads=rng.choice([4, 8, 12, 16]),
                    head_dim=64 if f32 else rng.choice([64, 64, 128]))
    if kind == "swin":
        grid = rng.choice([16, 24, 36, 48, 64])
        return dict(kind=kind, grid=grid, shells=shells(grid), geometry=geo,
                    window=rng.choice([4, 8]), heads=rng.choice([6, 8, 12]))
    if kind == "block":
        f32 = rng.random() < 0.4
        grid = rng.choice([12, 16, 24] if f32 else [12, 16, 24, 32, 48, 64])
        width = rng.choice([256, 512, 768, 1024])
        return dict(kind=kind, dtype="f32" if f32 else "bf16", grid=grid, shells=shells(grid),
                    geometry=geo, width=width, mlp=4 * width, tokens=log(64, 1370))
    if kind == "flow":
        grid = rng.choice([12, 16, 24, 32])
        width = rng.choice([512, 768, 1024])
        return dict(kind=kind, dtype="bf16", grid=grid, shells=shells(grid, 1, 0.2, 0.35),
                    geometry=geo, width=width, mlp=4 * width, blocks=rng.randint(4, 24),
                    tokens=log(64, 1370))
    return dict(kind="linear", dtype=rng.choice(["f32", "bf16"]), rows=log(200, 210000),
                cin=rng.choice([64, 128, 512, 768, 1024]), cout=rng.choice([64, 100, 256, 768, 1024]))


# ---- voxels ----------------------------------------------------------------

def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _ellipsoids(case):
    """Per item a list of (semi-axes, centre) in voxels of the case's grid."""
    rng = np.random.RandomState(case["geometry"])
    items = []
    for item in case["shells"].split(";"):
        parts = []
        for part in item.split(","):
            lo, hi = (float(v) for v in part.split("-"))
            axes = rng.uniform(lo, hi, 3)
            parts.append((axes, case["grid"] / 2.0 + np.floor(rng.uniform(0.0, 3.0, 3)) - 1.0))
        items.append(parts)
    return items


def _turn(seed):
    """A symmetry of the cube: axis order and which axes are mirrored."""
    r = random.Random(seed)
    order = [0, 1, 2]
    r.shuffle(order)
    return order, [r.random() < 0.5 for _ in range(3)]


def _inside(parts, grid, scale, xyz, turn):
    """Whether voxels xyz [n, 3] of the grid refined by `scale` lie in a shell."""
    order, mirrored = turn
    size = grid * scale
    cols = [(size - 1 - xyz[:, a]) if mirrored[a] else xyz[:, a] for a in range(3)]
    p = torch.stack([cols[order[a]] for a in range(3)], 1).double()
    hit = torch.zeros(xyz.shape[0], dtype=torch.bool, device=xyz.device)
    for axes, centre in parts:
        a = torch.tensor(axes * scale, dtype=torch.float64, device=xyz.device)
        c = torch.tensor(centre * scale, dtype=torch.float64, device=xyz.device)
        rho = (((p + 0.5 - c) / a) ** 2).sum(1).sqrt()
        hit |= (rho - 1.0).abs() * float(axes.min()) * scale < 1.0
    return hit


def _voxels(case, seed, dev):
    """int32 [n, 4] rows (batch, x, y, z), sorted."""
    g = case["grid"]
    ax = torch.arange(g, device=dev)
    xyz = torch.stack(torch.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    rows = []
    for b, parts in enumerate(_ellipsoids(case)):
        keep = xyz[_inside(parts, g, 1, xyz, _turn(seed))]
        rows.append(torch.cat([torch.full_like(keep[:, :1], b), keep], 1))
    return torch.cat(rows).to(torch.int32).contiguous()


def _children(coords, factor=2):
    """All children of the rows, parent by parent, child c at
    (c % f, c / f % f, c / f^2)."""
    n, cc = coords.shape[0], factor ** 3
    c = torch.arange(cc, device=coords.device)
    off = torch.stack([c % factor, c // factor % factor, c // (factor * factor)], 1)
    xyz = coords[:, None, 1:].long() * factor + off[None]
    b = coords[:, None, :1].long().expand(n, cc, 1)
    return torch.cat([b, xyz], 2).to(torch.int32)


def _surface_levels(case, seed, dev, levels):
    """The level coordinates of a surface refined level by level, and the
    subdivision flags [rows, 8] (+1 child kept, -1 dropped) between them."""
    coords = _voxels(case, seed, dev)
    items = _ellipsoids(case)
    out, guides = [coords], []
    for level in range(1, levels):
        kids = _children(coords)
        flat = kids.reshape(-1, 4)
        keep = torch.zeros(flat.shape[0], dtype=torch.bool, device=dev)
        for b, parts in enumerate(items):
            mine = flat[:, 0] == b
            keep[mine] = _inside(parts, case["grid"], 2 ** level, flat[mine][:, 1:].long(), _turn(seed))
        guides.append(torch.where(keep.reshape(-1, 8), 1.0, -1.0).float().contiguous())
        coords = flat[keep].contiguous()
        out.append(coords)
    return out, guides


def _keys(coords, dx=0, dy=0, dz=0):
    c = coords.long()
    return ((c[:, 0] * 4096 + c[:, 1] + dx + 1) * 4096 + c[:, 2] + dy + 1) * 4096 + c[:, 3] + dz + 1


def _neighbours(coords):
    """Yields (k, rows that have the neighbour, their neighbours' rows)."""
    base, perm = _keys(coords).sort()
    k = 0
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                want = _keys(coords, dx, dy, dz)
                at = torch.searchsorted(base, want).clamp_(max=base.shape[0] - 1)
                rows = (base[at] == want).nonzero()[:, 0]
                yield k, rows, perm[at[rows]]
                k += 1


def _pairs(coords):
    return sum(int(rows.shape[0]) for _, rows, _ in _neighbours(coords))


@lru_cache(maxsize=None)
def _counts(key):
    """(rows, neighbour pairs, coarse rows, coarse pairs) of a case's voxels."""
    coords = _voxels(dict(key), 0, _device())
    coarse = torch.unique(torch.cat([coords[:, :1], coords[:, 1:] // 2], 1), dim=0)
    return coords.shape[0], _pairs(coords), coarse.shape[0], _pairs(coarse)


@lru_cache(maxsize=None)
def _level_counts(key, levels):
    lv, _ = _surface_levels(dict(key), 0, _device(), levels)
    return [(c.shape[0], _pairs(c)) for c in lv]


def _key(case):
    return tuple((k, case[k]) for k in ("grid", "shells", "geometry"))


def _batch(case):
    return len(case["shells"].split(";"))


# ---- inputs ----------------------------------------------------------------

class _Rand:
    """Random tensors from the seed alone."""

    def __init__(self, seed, dev):
        self.dev = dev
        self.g = torch.Generator(device=dev).manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32, mean=0.0):
        return torch.randn(*shape, generator=self.g, device=self.dev).mul_(std).add_(mean).to(dtype)


def _block_tensors(r, dt, width, mlp, ctx):
    """A transformer block's tensors in P.BLOCK_WEIGHT_FIELDS order."""
    w = lambda o, i: r.normal(o, i, std=0.02, dtype=dt)  # noqa: E731
    b = lambda n: r.normal(n, std=0.02)  # noqa: E731
    gain = lambda n: r.normal(n, std=0.1, mean=1.0)  # noqa: E731
    return [b(6 * width), w(3 * width, width), b(3 * width), gain(width), gain(width),
            w(width, width), b(width), gain(width), b(width), w(width, width), b(width),
            w(2 * width, ctx), b(2 * width), gain(width), gain(width), w(width, width), b(width),
            None, None, w(mlp, width), b(mlp), w(width, mlp), b(width)]


def _decoder_blocks(r, dt, chans, predict):
    """[(kind, channels, out, hidden, tensors)] of a decoder with one ConvNeXt
    block per level."""
    out = []
    for i, c in enumerate(chans):
        out.append((P.PXS_DECODER_CONVNEXT, c, c, 4 * c, {
            "norm_weight": r.normal(c, std=0.1, mean=1.0), "norm_bias": r.normal(c, std=0.02),
            "conv1_weight": r.normal(27, c, c, std=(27 * c) ** -0.5, dtype=dt),
            "conv1_bias": r.normal(c, std=0.02),
            "mlp0_weight": r.normal(4 * c, c, std=c ** -0.5, dtype=dt),
            "mlp0_bias": r.normal(4 * c, std=0.02),
            "mlp2_weight": r.normal(c, 4 * c, std=0.02, dtype=dt),
            "mlp2_bias": r.normal(c, std=0.02)}))
        if i + 1 < len(chans):
            out.append((P.PXS_DECODER_C2S, c, chans[i + 1], 0,
                        _c2s_tensors(r, dt, c, chans[i + 1], predict)))
    return out


def _c2s_tensors(r, dt, c, o, predict):
    w = {"norm1_weight": r.normal(c, std=0.1, mean=1.0), "norm1_bias": r.normal(c, std=0.02),
         "conv1_weight": r.normal(27, 8 * o, c, std=(27 * c) ** -0.5, dtype=dt),
         "conv1_bias": r.normal(8 * o, std=0.02),
         "conv2_weight": r.normal(27, o, o, std=(27 * o) ** -0.5, dtype=dt),
         "conv2_bias": r.normal(o, std=0.02)}
    if predict:
        w["to_subdiv_weight"] = r.normal(8, c, std=c ** -0.5)
        w["to_subdiv_bias"] = r.normal(8, std=0.02)
    return w


def _inputs(case, seed):
    """The tensors of a case; `prepare` and `exact` both start from them."""
    dev = _device()
    r = _Rand(seed, dev)
    kind = case["kind"]
    dt = DTYPES[case.get("dtype", "bf16")]
    s = {}
    if "shells" in case and kind != "decoder":
        s["coords"] = _voxels(case, seed, dev)
    n = s["coords"].shape[0] if "coords" in s else 0
    if kind == "conv":
        ci, co = case["cin"], case["cout"]
        s["x"] = r.normal(n, ci, dtype=dt)
        s["w"] = r.normal(27, co, ci, std=(27 * ci) ** -0.5, dtype=dt)
        s["b"] = r.normal(co, std=0.02)
    elif kind == "unet":
        c1, c2 = case["c1"], case["c2"]
        s["x"] = r.normal(n, c1, dtype=dt)
        s["wa"] = r.normal(27, c1, c1, std=(2.0 / (27 * c1)) ** 0.5, dtype=dt)
        s["wb"] = r.normal(8, c2, c1, std=(2.0 / (8 * c1)) ** 0.5, dtype=dt)
        s["wc"] = r.normal(27, c2, c2, std=(2.0 / (27 * c2)) ** 0.5, dtype=dt)
        s["ba"], s["bb"], s["bc"] = (r.normal(c, std=0.02) for c in (c1, c2, c2))
    elif kind == "upsample":
        s["x"] = r.normal(n, case["cin"], dtype=dt)
        s["w"] = r.normal(27, 8 * case["out"], case["cin"], std=0.02, dtype=dt)
        s["b"] = r.normal(8 * case["out"], std=0.02)
    elif kind == "c2s":
        s["x"] = r.normal(n, case["channels"])
        s["w"] = _c2s_tensors(r, dt, case["channels"], case["out"], True)
        # As a trained decoder's hidden state does, x tells the children that
        # the refined surface meets from the others, each logit 0.5 or more
        # away from zero.
        w, b = s["w"]["to_subdiv_weight"].double(), s["w"]["to_subdiv_bias"].double()
        flags = _surface_levels(case, seed, dev, 2)[1][0].double()
        logits = s["x"].double() @ w.t() + b
        step = (flags * (logits.abs() + 0.5) - logits) @ torch.linalg.inv(w @ w.t()) @ w
        s["x"] = (s["x"].double() + step).float()
    elif kind == "decoder":
        chans = [int(c) for c in case["channels"].split(",")]
        s["chans"] = chans
        s["levels"], s["guides"] = _surface_levels(case, seed, dev, len(chans))
        s["coords"] = s["levels"][0]
        s["x"] = r.normal(s["coords"].shape[0], case["latent"])
        s["blocks"] = _decoder_blocks(r, dt, chans, False)
        s["io"] = [r.normal(chans[0], case["latent"], std=0.2), r.normal(chans[0], std=0.02),
                   r.normal(case["out"], chans[-1], std=0.1), r.normal(case["out"], std=0.02)]
    elif kind == "attn":
        lens = [int(v) for v in case["lengths"].split(",")]
        n, c = sum(lens), case["heads"] * case["head_dim"]
        s["x"] = r.normal(n, c, dtype=dt)
        s["wqkv"], s["bqkv"] = r.normal(3 * c, c, std=0.02, dtype=dt), r.normal(3 * c, std=0.02)
        s["wo"], s["bo"] = r.normal(c, c, std=0.02, dtype=dt), r.normal(c, std=0.02)
        s["gq"], s["gk"] = r.normal(c, std=0.1, mean=1.0), r.normal(c, std=0.1, mean=1.0)
        s["cu"] = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=dev)
    elif kind == "swin":
        c = 64 * case["heads"]
        s["x"] = r.normal(n, c, dtype=dt)
        s["layers"] = [(r.normal(3 * c, c, std=0.02, dtype=dt), r.normal(3 * c, std=0.02),
                        r.normal(c, c, std=0.02, dtype=dt), r.normal(c, std=0.02)) for _ in range(2)]
    elif kind in ("block", "flow"):
        c, t = case["width"], case["tokens"]
        count = case.get("blocks", 1)
        s["blocks"] = [_block_tensors(r, dt, c, case["mlp"], c) for _ in range(count)]
        s["ctx"] = r.normal(t, c, dtype=dt)
        s["ctx_off"] = torch.tensor([0, t], dtype=torch.int64, device=dev)
        s["cu"] = torch.tensor([0, n], dtype=torch.int64, device=dev)
        if kind == "block":
            s["hidden"] = r.normal(n, c)
            s["time_mod"] = r.normal(1, 6 * c, std=0.2)
        else:
            s["x"] = r.normal(n, 8)
            s["t"] = torch.rand(1, generator=r.g, device=dev) * 1000.0
            s["io"] = [r.normal(c, 8, std=0.2), r.normal(c, std=0.02), r.normal(c, 256, std=0.02),
                       r.normal(c, std=0.02), r.normal(c, c, std=0.02), r.normal(c, std=0.02),
                       r.normal(6 * c, c, std=0.02), r.normal(6 * c, std=0.02),
                       r.normal(8, c, std=0.02), r.normal(8, std=0.02)]
    else:
        s["x"] = r.normal(case["rows"], case["cin"], dtype=dt)
        s["w"] = r.normal(case["cout"], case["cin"], std=case["cin"] ** -0.5, dtype=dt)
        s["b"] = r.normal(case["cout"], std=0.02)
    return s


_PX = None


def prepare(case, seed):
    global _PX
    if _PX is None:
        _PX = P.Pxs()
    px = _PX
    s = _inputs(case, seed)
    s["case"], s["px"] = case, px
    kind = case["kind"]
    if "grid" in case:
        s["shape"], s["batch"] = (case["grid"],) * 3, _batch(case)
    if kind == "unet":
        # Kept over the steps of a loop: the tagged grid, the stride-2
        # workspace, the coarse grid, and the coarse row count.
        s["fine"] = px.tagged_grid(s["batch"], s["shape"])
        s["ws"] = px.s2_tagged_workspace(s["batch"], s["shape"])
        cells = px.lib.pxs_voxel_grid_bytes(s["batch"], *(((e + 1) // 2) for e in s["shape"])) // 4
        s["coarse"] = torch.empty(cells, dtype=torch.int32, device=_device())
        s["gen"] = 0
        c = s["coords"]
        s["m"] = int(torch.unique(torch.cat([c[:, :1], c[:, 1:] // 2], 1), dim=0).shape[0])
    elif kind == "c2s":
        s["weights"] = P.decoder_block_weights(s["w"])
    elif kind == "decoder":
        s["native"] = [P.DecoderBlock(k, c, o, h, P.decoder_block_weights(w))
                       for k, c, o, h, w in s["blocks"]]
        s["cfg"] = P.decoder_config(case["latent"], case["out"], 1e-6, False, s["chans"],
                                    [1] * len(s["chans"]))
        # every level but the last may grow eightfold
        s["max_rows"] = 8 * max(c.shape[0] for c in s["levels"][:-1])
        s.pop("levels")
    elif kind in ("block", "flow"):
        c, h = case["width"], case["width"] // 64
        native = [P.block_weights(t) for t in s["blocks"]]
        if kind == "block":
            s["native"] = native[0]
            s["cfg"] = P.BlockConfig(c, h, case["mlp"], c, 0, 1e-6, 1.0, 10000.0, 1, 1, 1, 0)
        else:
            s["array"] = (P.BlockWeights * len(native))(*native)
            s["native"] = P.FlowWeights(*[t.data_ptr() for t in s["io"]], s["array"])
            s["cfg"] = P.FlowConfig(8, 8, c, c, len(native), h, 0, case["mlp"], 1e-6, 1.0, 10000.0,
                                    1, 1, 0)
    return s


# ---- one pass --------------------------------------------------------------

def run(s):
    case, px = s["case"], s["px"]
    kind = case["kind"]
    if kind == "conv":
        if case["lookup"] == "grid":
            grid = px.grid_build(s["coords"], s["batch"], s["shape"])
            return px.subm_conv3d_grid(s["x"], s["w"], s["b"], s["coords"], s["batch"], s["shape"],
                                       grid)
        find = px.neighbor_map if case["lookup"] == "hash" else px.neighbor_map_bricks
        nbr, masks = find(s["coords"])
        return nbr, masks, px.subm_conv3d(s["x"], s["w"], s["b"], nbr, masks)
    if kind == "unet":
        b, shape, m = s["batch"], s["shape"], s["m"]
        if s["gen"] == 255:  # generations between two resets
            px._check(px.lib.pxs_voxel_grid_tagged_reset(s["fine"].data_ptr(), b, *shape,
                                                         px.stream()), "reset")
            px._check(px.lib.pxs_downsample_s2_tagged_workspace_reset(
                s["ws"].data_ptr(), b, *shape, px.stream()), "reset")
            s["gen"] = 0
        s["gen"] += 1
        px.s2_tagged_insert(s["coords"], b, shape, s["fine"], s["gen"], s["ws"])
        ya, oc, child, count = px.subm_conv3d_grid_s2_emit(
            s["x"], s["wa"], s["ba"], s["coords"], b, shape, s["fine"], s["gen"], s["coarse"], s["ws"])
        yb = px.sparse_conv3d_s2(ya, s["wb"], s["bb"], child, m)
        half = tuple((e + 1) // 2 for e in shape)
        yc = px.subm_conv3d_grid(yb, s["wc"], s["bc"], oc[:m], b, half, s["coarse"])
        return ya, yb, yc, oc[:m], child[:, :m], count
    if kind == "upsample":
        grid = px.grid_build(s["coords"], s["batch"], s["shape"])
        packed = px.subm_conv3d_grid(s["x"], s["w"], s["b"], s["coords"], s["batch"], s["shape"],
                                     grid)
        return px.channel_to_spatial(s["coords"], packed)
    if kind == "c2s":
        return px.resblock_c2s(s["coords"], s["x"], case["out"], 1e-6, s["weights"],
                               CODES[case["dtype"]], pred_subdiv=True)
    if kind == "decoder":
        oc, y, rows, _ = px.slat_decoder_forward(
            CODES[case["dtype"]], s["cfg"], *s["io"], s["native"], s["coords"], s["x"],
            guide=s["guides"], max_rows=s["max_rows"])
        return oc, y
    if kind == "attn":
        h, d = case["heads"], case["head_dim"]
        qkv = px.linear(s["x"], s["wqkv"], s["bqkv"])
        q, k, v = px.qkv_prepare(qkv, h, d, s["gq"], s["gk"])
        o = px.varlen_attention(q, k, v, s["cu"], s["cu"], h, d, d ** -0.5)
        return px.linear(o, s["wo"], s["bo"])
    if kind == "swin":
        h = case["heads"]
        c, x, maps = 64 * h, s["x"], []
        for i, (wqkv, bqkv, wo, bo) in enumerate(s["layers"]):
            fwd, bwd, cu, nseg = px.window_partition(s["coords"], s["batch"], s["shape"],
                                                     case["window"], i * case["window"] // 2,
                                                     sync=False)
            qkv = px.linear(x, wqkv, bqkv)
            o = px.varlen_attention(qkv[:, :c], qkv[:, c:2 * c], qkv[:, 2 * c:], cu, cu, h, 64,
                                    0.125, row_map=fwd, nseg=nseg)
            x = px.linear(o, wo, bo)
            maps += [fwd, bwd, cu]
        return [x] + maps
    if kind == "block":
        return px.transformer_block(s["cfg"], s["native"], s["coords"], 1, s["cu"],
                                    s["hidden"].clone(), s["time_mod"], s["ctx"], s["ctx_off"])
    if kind == "flow":
        return px.slat_flow_forward(s["cfg"], s["native"], s["coords"], 1, s["cu"], s["x"], s["t"],
                                    s["ctx"], s["ctx_off"])
    return px.linear(s["x"], s["w"], s["b"])


# ---- the work a pass cannot do without --------------------------------------

def _block_work(n, t, c, mlp, e):
    flops = 4.0 * n * n * c + 4.0 * n * t * c + 2.0 * n * c * (6 * c + 2 * mlp) + 4.0 * t * c * c
    return (8 * c * c + 2 * c * mlp) * e + t * c * e, flops


def work(case):
    kind = case["kind"]
    e = SIZE[case.get("dtype", "bf16")]
    if kind == "linear":
        n, ci, co = case["rows"], case["cin"], case["cout"]
        return {"bytes": (n * (ci + co) + ci * co) * e, "flops": 2.0 * n * ci * co}
    if kind == "attn":
        lens = [int(v) for v in case["lengths"].split(",")]
        n, c = sum(lens), case["heads"] * case["head_dim"]
        return {"bytes": (2 * n * c + 4 * c * c) * e,
                "flops": 8.0 * n * c * c + 4.0 * sum(v * v for v in lens) * c}
    if kind == "decoder":
        chans = [int(c) for c in case["channels"].split(",")]
        lv = _level_counts(_key(case), len(chans))
        flops = 2.0 * lv[0][0] * case["latent"] * chans[0] + 2.0 * lv[-1][0] * chans[-1] * case["out"]
        weights = 0
        for i, (c, (rows, pairs)) in enumerate(zip(chans, lv)):
            flops += 2.0 * pairs * c * c + 16.0 * rows * c * c
            weights += 35 * c * c
            if i + 1 < len(chans):
                o = chans[i + 1]
                flops += 16.0 * pairs * c * o + 2.0 * lv[i + 1][1] * o * o
                weights += 27 * (8 * c * o + o * o)
        moved = lv[0][0] * (16 + 4 * case["latent"]) + lv[-1][0] * (16 + 4 * case["out"])
        moved += sum(32 * rows for rows, _ in lv[:-1])
        return {"bytes": moved + weights * e, "flops": flops}
    n, pairs, m, coarse_pairs = _counts(_key(case))
    if kind == "conv":
        ci, co = case["cin"], case["cout"]
        moved = n * 16 + (n * (ci + co) + 27 * ci * co) * e
        return {"bytes": moved + (0 if case["lookup"] == "grid" else 112 * n),
                "flops": 2.0 * pairs * ci * co}
    if kind == "unet":
        c1, c2 = case["c1"], case["c2"]
        weights = 27 * c1 * c1 + 8 * c1 * c2 + 27 * c2 * c2
        return {"bytes": n * 16 + m * 48 + (2 * n * c1 + 2 * m * c2 + weights) * 2,
                "flops": 2.0 * (pairs * c1 * c1 + n * c1 * c2 + coarse_pairs * c2 * c2)}
    if kind == "upsample":
        ci, o = case["cin"], case["out"]
        return {"bytes": n * (16 + 8 * 16) + (n * (ci + 8 * o) + 27 * 8 * o * ci) * 2,
                "flops": 2.0 * pairs * ci * 8 * o}
    if kind == "c2s":
        c, o = case["channels"], case["out"]
        kids, kid_pairs = _level_counts(_key(case), 2)[1]
        return {"bytes": n * (16 + 4 * c + 32) + kids * (16 + 4 * o) + 27 * (8 * c * o + o * o) * e,
                "flops": 2.0 * (8 * n * c + 8 * pairs * c * o + kid_pairs * o * o)}
    if kind == "swin":
        c, w = 64 * case["heads"], case["window"]
        flops = 2 * 8.0 * n * c * c
        for shift in (0, w // 2):
            cells = (_voxels(case, 0, _device()) + torch.tensor([0] + [shift] * 3, device=_device()))
            cells[:, 1:] //= w
            lens = torch.unique(cells, dim=0, return_counts=True)[1].double()
            flops += 4.0 * float((lens * lens).sum()) * c
        return {"bytes": n * 16 + (2 * n * c + 8 * c * c) * 2 + 2 * n * 8, "flops": flops}
    c, t = case["width"], case["tokens"]
    weights, flops = _block_work(n, t, c, case["mlp"], e)
    if kind == "block":
        return {"bytes": weights + n * (16 + 8 * c), "flops": flops}
    count = case["blocks"]
    return {"bytes": count * weights + n * (16 + 64) + 7 * c * c * 4, "flops": count * flops}


# ---- tolerances --------------------------------------------------------------

def tolerance(case):
    """About four times the distance to the 64-bit result; whole numbers
    (coordinates, maps, permutations) stay the same."""
    kind, f32 = case["kind"], case.get("dtype") == "f32"
    if f32:
        return {"rel": {"block": 1e-6, "attn": 4e-6}.get(kind, 2.5e-6)}
    return {"rel": {"block": 1.5e-3, "flow": 6e-3, "decoder": 2.5e-2}.get(kind, 1e-2)}


# ---- the same outputs in 64 bits ---------------------------------------------

def _linear64(x, w, b):
    return x.double() @ w.double().t() + b.double()


def _conv64(coords, x, w, b):
    x = x.double()
    y = b.double().repeat(x.shape[0], 1)
    for k, rows, src in _neighbours(coords):
        if rows.shape[0]:
            y[rows] += x[src] @ w[k].double().t()
    return y


def _norm64(x, eps, gamma=None, beta=None):
    x = x - x.mean(1, keepdim=True)
    x = x / (x.pow(2).mean(1, keepdim=True) + eps).sqrt()
    return x if gamma is None else x * gamma.double() + beta.double()


def _rms64(x, heads, gamma):
    n, c = x.shape
    x = x.reshape(n, heads, c // heads)
    x = x / x.pow(2).sum(2, keepdim=True).sqrt().clamp(min=1e-12) * (c // heads) ** 0.5
    return x.reshape(n, c) * gamma.double()


def _rope64(x, heads, coords):
    n, c = x.shape
    pairs = c // heads // 2
    f = pairs // 3
    freq = 10000.0 ** (-torch.arange(f, dtype=torch.float64, device=x.device) / f)
    phase = (coords[:, 1:].double()[:, :, None] * freq).reshape(n, 1, 3 * f)
    phase = torch.nn.functional.pad(phase, (0, pairs - 3 * f))
    e, o = x.reshape(n, heads, pairs, 2).unbind(3)
    cos, sin = phase.cos(), phase.sin()
    return torch.stack([e * cos - o * sin, e * sin + o * cos], 3).reshape(n, c)


def _attention64(q, k, v, cu_q, cu_k, heads):
    n, c = q.shape
    d = c // heads
    out = torch.empty_like(q)
    for a, b, ka, kb in zip(cu_q[:-1], cu_q[1:], cu_k[:-1], cu_k[1:]):
        for h in range(heads):
            cols = slice(h * d, (h + 1) * d)
            kh, vh = k[ka:kb, cols].t().contiguous(), v[ka:kb, cols].contiguous()
            for r in range(a, b, 4096):
                p = torch.softmax((q[r:min(b, r + 4096), cols] @ kh) * d ** -0.5, 1)
                out[r:min(b, r + 4096), cols] = p @ vh
    return out


def _block64(t, h, coords, ctx, time_mod, heads):
    (mod, wqkv, bqkv, gq, gk, wo, bo, n2w, n2b, wcq, bcq, wkv, bkv, gcq, gck, wco, bco, _, _, w0, b0,
     w2, b2) = t
    n, c = h.shape
    m = mod.double() + time_mod[0].double()
    x = _norm64(h, 1e-6) * (1 + m[c:2 * c]) + m[:c]
    q, k, v = _linear64(x, wqkv, bqkv).split(c, 1)
    q, k = (_rope64(_rms64(a, heads, g), heads, coords) for a, g in ((q, gq), (k, gk)))
    h = h + _linear64(_attention64(q, k, v, [0, n], [0, n], heads), wo, bo) * m[2 * c:3 * c]
    x = _norm64(h, 1e-6, n2w, n2b)
    q = _rms64(_linear64(x, wcq, bcq), heads, gcq)
    k, v = _linear64(ctx, wkv, bkv).split(c, 1)
    k = _rms64(k, heads, gck)
    h = h + _linear64(_attention64(q, k, v, [0, n], [0, ctx.shape[0]], heads), wco, bco)
    x = _norm64(h, 1e-6) * (1 + m[4 * c:5 * c]) + m[3 * c:4 * c]
    x = torch.nn.functional.gelu(_linear64(x, w0, b0), approximate="tanh")
    return h + _linear64(x, w2, b2) * m[5 * c:]


def _c2s64(coords, x, w, out, keep):
    """The up-block with the children `keep` [rows, 8] -> (coords, features)."""
    silu = torch.nn.functional.silu
    n = x.shape[0]
    y = _conv64(coords, silu(_norm64(x, 1e-6, w["norm1_weight"], w["norm1_bias"])),
                w["conv1_weight"], w["conv1_bias"]).reshape(n, 8, out)[keep]
    oc = _children(coords)[keep]
    skip = x.reshape(n, 8, -1)[keep]
    y = _conv64(oc, silu(_norm64(y, 1e-6)), w["conv2_weight"], w["conv2_bias"])
    return oc, y + skip.repeat_interleave(out // skip.shape[1], 1)


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "conv":
        y = _conv64(s["coords"], s["x"], s["w"], s["b"])
        if case["lookup"] == "grid":
            return y
        n = s["coords"].shape[0]
        nbr = torch.full((27, n), n, dtype=torch.int32, device=y.device)
        masks = torch.zeros(n, dtype=torch.int32, device=y.device)
        for k, rows, src in _neighbours(s["coords"]):
            nbr[k, rows] = src.to(torch.int32)
            masks[rows] |= 1 << k
        return nbr, masks, y
    if kind == "unet":
        c = s["coords"]
        coarse, parent = torch.unique(torch.cat([c[:, :1], c[:, 1:] // 2], 1), dim=0,
                                      return_inverse=True)
        m = coarse.shape[0]
        slot = c[:, 1] % 2 + 2 * (c[:, 2] % 2) + 4 * (c[:, 3] % 2)
        child = torch.full((8, m), -1, dtype=torch.int32, device=c.device)
        child[slot.long(), parent] = torch.arange(c.shape[0], dtype=torch.int32, device=c.device)
        ya = _conv64(c, s["x"], s["wa"], s["ba"])
        yb = s["bb"].double().repeat(m, 1)
        for k in range(8):
            rows = (slot == k).nonzero()[:, 0]
            yb[parent[rows]] += ya[rows] @ s["wb"][k].double().t()
        yc = _conv64(coarse, yb, s["wc"], s["bc"])
        return ya, yb, yc, coarse, child, torch.tensor([m], device=c.device)
    if kind == "upsample":
        packed = _conv64(s["coords"], s["x"], s["w"], s["b"])
        return _children(s["coords"]).reshape(-1, 4), packed.reshape(-1, case["out"])
    if kind == "c2s":
        logits = _linear64(s["x"], s["w"]["to_subdiv_weight"], s["w"]["to_subdiv_bias"])
        return *_c2s64(s["coords"], s["x"].double(), s["w"], case["out"], logits > 0), logits
    if kind == "decoder":
        x = _linear64(s["x"], s["io"][0], s["io"][1])
        coords, guides = s["coords"], iter(s["guides"])
        for k, c, o, _, w in s["blocks"]:
            if k == P.PXS_DECODER_CONVNEXT:
                y = _norm64(_conv64(coords, x, w["conv1_weight"], w["conv1_bias"]), 1e-6,
                            w["norm_weight"], w["norm_bias"])
                y = torch.nn.functional.silu(_linear64(y, w["mlp0_weight"], w["mlp0_bias"]))
                x = x + _linear64(y, w["mlp2_weight"], w["mlp2_bias"])
            else:
                coords, x = _c2s64(coords, x, w, o, next(guides) > 0)
        return coords, _linear64(_norm64(x, 1e-5), s["io"][2], s["io"][3])
    if kind == "attn":
        h = case["heads"]
        q, k, v = _linear64(s["x"], s["wqkv"], s["bqkv"]).chunk(3, 1)
        cu = s["cu"].tolist()
        o = _attention64(_rms64(q, h, s["gq"]), _rms64(k, h, s["gk"]), v, cu, cu, h)
        return _linear64(o, s["wo"], s["bo"])
    if kind == "swin":
        coords, g, w = s["coords"].long(), case["grid"], case["window"]
        n = coords.shape[0]
        x, maps = s["x"].double(), []
        for i, (wqkv, bqkv, wo, bo) in enumerate(s["layers"]):
            shift = i * w // 2
            side = (g + shift + w - 1) // w
            cell = (coords[:, 1:] + shift) // w
            wid = ((coords[:, 0] * side + cell[:, 0]) * side + cell[:, 1]) * side + cell[:, 2]
            _, fwd = wid.sort(stable=True)
            bwd = torch.empty_like(fwd)
            bwd[fwd] = torch.arange(n, device=fwd.device)
            lens = torch.unique(wid, return_counts=True)[1]
            cu = torch.cat([lens.new_zeros(1), lens.cumsum(0)])
            q, k, v = _linear64(x, wqkv, bqkv)[fwd].chunk(3, 1)
            o = torch.empty_like(q)
            edges = cu.tolist()
            h = case["heads"]
            for a, b in zip(edges[:-1], edges[1:]):
                qh, kh, vh = (t[a:b].reshape(b - a, h, 64).transpose(0, 1).contiguous()
                              for t in (q, k, v))
                p = torch.softmax(qh @ kh.transpose(1, 2).contiguous() * 0.125, 2)
                o[a:b] = (p @ vh).transpose(0, 1).reshape(b - a, 64 * h)
            x = torch.empty_like(o)
            x[fwd] = _linear64(o, wo, bo)
            full = torch.full((min(n, _batch(case) * side ** 3) + 1,), n, device=cu.device)
            full[:cu.shape[0]] = cu
            maps += [fwd.to(torch.int32), bwd.to(torch.int32), full]
        return [x] + maps
    if kind == "block":
        return _block64(s["blocks"][0], s["hidden"].double(), s["coords"], s["ctx"], s["time_mod"],
                        case["width"] // 64)
    if kind == "flow":
        wi, bi, w0, b0, w2, b2, wm, bm, wo, bo = s["io"]
        silu = torch.nn.functional.silu
        freq = torch.exp(-math.log(10000.0) / 128
                         * torch.arange(128, dtype=torch.float64, device=wi.device))
        arg = s["t"].double()[:, None] * freq
        emb = torch.cat([arg.cos(), arg.sin()], 1)
        mod = _linear64(silu(_linear64(silu(_linear64(emb, w0, b0)), w2, b2)), wm, bm)
        h = _linear64(s["x"], wi, bi)
        for t in s["blocks"]:
            h = _block64(t, h, s["coords"], s["ctx"], mod, case["width"] // 64)
        return _linear64(_norm64(h, 1e-5), wo, bo)
    return _linear64(s["x"], s["w"], s["b"])
