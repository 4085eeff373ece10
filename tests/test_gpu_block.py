"""Device-resident transformer block and SLat-flow forward (pxs_transformer_block,
pxs_slat_flow_forward) against the compiled reference's vectors and the oracle.

fp32: within 1e-5 (max|g - r| / max|r|).  bf16 GEMM operands with fp32
accumulation and an fp32 residual stream: within 1e-2 relative L2, against the
oracle run in fp32 on the same bf16-rounded weights and inputs.
"""

from pathlib import Path

import numpy as np
import pytest
import torch

import oracle as O
import pxs
import workloads as W
from fixtures import flow_case
from gpu_common import assert_bf16, assert_fp32, dev, host, rel_l2, t32, ti32, ti64

pytestmark = pytest.mark.gpu
GOLD = Path(__file__).resolve().parent / "golden"


@pytest.fixture(scope="module")
def px():
    return pxs.Pxs()


@pytest.fixture(scope="module")
def orc():
    return O.Oracle()


def block_cfg(C, H, M, CC, PC, use_proj, eps=1e-6):
    return pxs.BlockConfig(C, H, M, CC, PC, eps, 1.0, 10000.0, 1, 1, 1, 1 if use_proj else 0)


def device_weights(ws, dtype):
    """Host arrays -> device tensors; linear weights in dtype, the rest fp32."""
    out = []
    for i, w in enumerate(ws):
        if w is None:
            out.append(None)
            continue
        t = t32(w)
        out.append(t.to(dtype) if (i in pxs.BLOCK_LINEAR_WEIGHTS and dtype != torch.float32) else t)
    return out


def bf16_round(ws):
    return [None if w is None else (W.bf16_round(w) if i in pxs.BLOCK_LINEAR_WEIGHTS else w)
            for i, w in enumerate(ws)]


@pytest.mark.parametrize("proj", [True, False])
def test_block_fp32_reference_vectors(px, proj):
    v = dict(np.load(GOLD / "ref_vectors.npz"))
    ws = [v[f"blk_w{i}"] for i in range(23)]
    if not proj:
        ws[17] = ws[18] = None
    dws = device_weights(ws, torch.float32)
    cfg = block_cfg(32, 4, 64, 6, 5, proj)
    coords = ti32(v["blk_coords"])
    cu = px.batch_cu_seqlens(coords, 2)
    hidden = t32(v["blk_x"]).clone()
    px.transformer_block(cfg, pxs.block_weights(dws), coords, 2, cu, hidden, t32(v["blk_tmod"]),
                         t32(v["blk_ctx"]), ti64(v["blk_ctx_off"]),
                         projected=t32(v["blk_proj"]) if proj else None)
    assert_fp32(host(hidden), v["blk_out"] if proj else v["blk_out_noproj"],
                what=f"block fp32 proj={proj}")


def run_flow(px, case, dtype):
    C, H, M, CC = case["C"], case["H"], case["M"], case["CC"]
    nb = len(case["blocks"])
    cfg = pxs.FlowConfig(case["dims"][0], case["dims"][2], C, CC, nb, H, 0, M, 1e-6, 1.0, 10000.0,
                         1, 1, 0)
    fw_dev = [t32(a) for a in case["fw"]]
    blk_dev = [device_weights(ws, dtype) for ws in case["blocks"]]
    arr = (pxs.BlockWeights * max(nb, 1))(*[pxs.block_weights(b) for b in blk_dev])
    weights = pxs.FlowWeights(*[a.data_ptr() for a in fw_dev], arr)
    coords = ti32(case["coords"])
    bsz = len(case["ctx_off"]) - 1
    cu = px.batch_cu_seqlens(coords, bsz)
    ctx = t32(case["ctx"]).to(dtype)
    out = px.slat_flow_forward(cfg, weights, coords, bsz, cu, t32(case["x"]), t32(case["t"]), ctx,
                               ti64(case["ctx_off"]))
    torch.cuda.synchronize()
    return host(out)


def oracle_flow(orc, case, bf16):
    blocks = [bf16_round(ws) for ws in case["blocks"]] if bf16 else case["blocks"]
    ctx = W.bf16_round(case["ctx"]) if bf16 else case["ctx"]
    return orc.slat_flow_forward(case["coords"], len(case["ctx_off"]) - 1, case["x"], case["t"],
                                 ctx, case["ctx_off"], case["dims"], [1e-6, 1.0, 10000.0],
                                 case["fw"], blocks)


def test_flow_fp32_small(px, orc):
    """Two blocks, C=64 (2 heads x 32), two batches of ~300 voxels; fp32 end to end."""
    case = flow_case(31, [[(4.0, 6.0)], [(3.0, 5.0)]], 16, 64, 2, 2, 7)
    print(f"flow fp32: n={case['n']}", flush=True)
    got = run_flow(px, case, torch.float32)
    ref = oracle_flow(orc, case, bf16=False)
    assert_fp32(got, ref, what="flow fp32")


def test_flow_bf16_reduced_config(px, orc):
    """The SLat-flow step at reduced size: 2 blocks of width 1024 (16 heads x 64,
    MLP 4096), 1,904 voxels in 2 batches, 137 context tokens each; bf16 GEMMs."""
    case = flow_case(32, [[(5.0, 7.0)], [(4.0, 6.0)]], 32, 1024, 16, 2, 137)
    print(f"flow bf16: n={case['n']}", flush=True)
    got = run_flow(px, case, torch.bfloat16)
    ref = oracle_flow(orc, case, bf16=True)
    assert np.isfinite(got).all()
    assert_bf16(got, ref, what="flow bf16 reduced")


def test_flow_bf16_full_depth(px, orc):
    """The SLat-flow step at its full depth and width: 24 blocks of width 1024
    (16 heads x 64, MLP 4096), 864 voxels in 2 batches, 137 context tokens
    each; bf16 GEMMs against the oracle's fp32 forward on the same
    bf16-rounded weights, so rounding that compounds over the 24 residual
    updates is held to the same 1e-2 relative L2 as one block."""
    case = flow_case(33, [[(4.0, 6.0)], [(3.0, 5.0)]], 24, 1024, 16, 24, 137)
    print(f"flow bf16 24 blocks: n={case['n']}", flush=True)
    got = run_flow(px, case, torch.bfloat16)
    ref = oracle_flow(orc, case, bf16=True)
    assert np.isfinite(got).all()
    print(f"flow bf16 24 blocks: rel L2 {rel_l2(got, ref):.3e}", flush=True)
    assert_bf16(got, ref, what="flow bf16 24 blocks")


def test_block_fp32_wide_heads(px, orc):
    """A block with 128-wide heads (C = 256, 2 heads; RoPE, q/k RMS norms,
    cross-attention), fp32, against the oracle block
    (src/sparse_transformer.cpp:138-292); the reference allows any head width."""
    from test_gpu_configs import flow_block_weights, normal
    rng = np.random.default_rng(94)
    coords = W.shell_coords(12, [[(3.0, 5.0)], [(2.0, 4.0)]], 94)
    n, C, H, M, CC, T = coords.shape[0], 256, 2, 512, 64, 9
    ws = flow_block_weights(rng, C, M, CC)
    x = normal(rng, (n, C))
    tmod = normal(rng, (2, 6 * C), 0.3)
    ctx = normal(rng, (2 * T, CC))
    off = np.array([0, T, 2 * T], np.int64)
    print(f"[block wide heads] n={n} head_dim={C // H}", flush=True)
    c = ti32(coords)
    hidden = t32(x).clone()
    dws = device_weights(ws, torch.float32)  # kept alive: the struct holds raw pointers
    px.transformer_block(block_cfg(C, H, M, CC, 0, False), pxs.block_weights(dws), c, 2,
                         px.batch_cu_seqlens(c, 2), hidden, t32(tmod), t32(ctx), ti64(off))
    ref = orc.transformer_block(coords, 2, x, tmod, ctx, off, [C, H, M, CC, 0, 1, 1, 1, 0],
                                [1e-6, 1.0, 10000.0], ws)
    assert_fp32(host(hidden), ref, what="block wide heads")


@pytest.mark.parametrize("C,rows,M,PC", [(256, 1, 512, 0), (512, 130, 1024, 0), (768, 129, 520, 36),
                                         (1024, 260, 1024, 256)])
def test_block_residual_linears_split_over_k(px, orc, C, rows, M, PC):
    """Blocks of few rows: the residual linears whose K is long enough run split
    over K, with the residual's update and the next norm in one pass (each
    width of that pass; MLP-2 with a ragged last K chunk; a projection that
    is split and one that is not), fp32, against the oracle block."""
    from test_gpu_configs import flow_block_weights, normal
    rng = np.random.default_rng(95)
    coords = W.shell_coords(16, [[(4.0, 6.0)], [(3.0, 5.0)]], 95)
    keep = np.sort(rng.permutation(coords.shape[0])[:rows])
    coords = np.ascontiguousarray(coords[keep])
    H, CC, T = C // 64, 64, 9
    ws = flow_block_weights(rng, C, M, CC)
    proj = None
    if PC:
        ws[17], ws[18] = normal(rng, (C, PC), 0.02), normal(rng, (C,), 0.02)
        proj = normal(rng, (rows, PC))
    x = normal(rng, (rows, C))
    tmod = normal(rng, (2, 6 * C), 0.3)
    ctx = normal(rng, (2 * T, CC))
    off = np.array([0, T, 2 * T], np.int64)
    print(f"[block split] rows={rows} C={C} M={M} PC={PC}", flush=True)
    c = ti32(coords)
    hidden = t32(x).clone()
    dws = device_weights(ws, torch.float32)  # kept alive: the struct holds raw pointers
    px.transformer_block(block_cfg(C, H, M, CC, PC, PC > 0), pxs.block_weights(dws), c, 2,
                         px.batch_cu_seqlens(c, 2), hidden, t32(tmod), t32(ctx), ti64(off),
                         projected=t32(proj) if PC else None)
    ref = orc.transformer_block(coords, 2, x, tmod, ctx, off, [C, H, M, CC, PC, 1, 1, 1, int(PC > 0)],
                                [1e-6, 1.0, 10000.0], ws, projected=proj)
    assert_fp32(host(hidden), ref, what="block split")


# Rows on both sides of the one-pass line (170 tiles of 128 x 128), ragged ones,
# and each split count (4, 3, 2 at width 256: 48, 80 and 170 tiles).
@pytest.mark.parametrize("C,rows,M,PC", [(1024, 130, 1024, 0), (256, 1, 1024, 1024), (256, 3000, 1024, 0),
                                         (256, 5120, 1024, 1024), (256, 10880, 1024, 0), (256, 10881, 1024, 0),
                                         (512, 700, 2048, 2048)])
@pytest.mark.parametrize("part", ["self", "cross", "projection", "mlp"])
def test_block_bf16_residual_linears_split_over_k(px, C, rows, M, PC, part):
    """One residual linear of a bf16 block at a time (the others' weights zero),
    against the block made of single ops, whose linears run in one pass: the
    fp32 update differs by the order of its sums only."""
    if part == "projection" and not PC:
        pytest.skip("no projection in this block")
    H, T, bf = C // 64, 12, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(rows + C)
    rand = lambda *s, std=1.0: torch.randn(*s, device="cuda", generator=g) * std  # noqa: E731
    i = torch.arange(rows, device="cuda")
    batch = 2 if rows > 1 else 1
    c = torch.stack([i * batch // rows, i // 256, i // 16 % 16, i % 16], 1).to(torch.int32)
    cu = px.batch_cu_seqlens(c, batch)
    sizes = [6 * C, 3 * C * C, 3 * C, C, C, C * C, C, C, C, C * C, C, 2 * C * C, 2 * C, C, C, C * C, C,
             C * PC, C if PC else 0, M * C, M, C * M, C]
    ws = [rand(n, std=0.03) if n else None for n in sizes]
    for k in (3, 4, 7, 13, 14):
        ws[k] = ws[k] + 1.0
    for name, (wi, bi) in {"self": (5, 6), "cross": (15, 16), "projection": (17, 18), "mlp": (21, 22)}.items():
        if name != part and ws[wi] is not None:
            ws[wi], ws[bi] = ws[wi] * 0, ws[bi] * 0
    ws = [w.to(bf) if w is not None and k in pxs.BLOCK_LINEAR_WEIGHTS else w for k, w in enumerate(ws)]
    x, tm = rand(rows, C), rand(batch, 6 * C, std=0.3)
    ctx, off = rand(batch * T, C).to(bf), ti64(np.arange(batch + 1) * T)
    proj = rand(rows, PC).to(bf) if PC else None
    print(f"[block bf16 split] rows={rows} C={C} M={M} PC={PC} {part}", flush=True)
    got = x.clone()
    px.transformer_block(block_cfg(C, H, M, C, PC, PC > 0), pxs.block_weights(ws), c, batch, cu, got, tm,
                         ctx, off, projected=proj)
    ref, w2 = x.clone(), lambda k, n: ws[k].view(n, -1)  # noqa: E731
    if part == "self":
        xm = px.layer_norm_modulate(ref, 1e-6, c, ws[0], tm, 0, out_dtype=bf)
        q, k, v = px.qkv_prepare(px.linear(xm, w2(1, 3 * C), ws[2]), H, 64, ws[3], ws[4], c)
        att = px.varlen_attention(q, k, v, cu, cu, H, 64, 0.125)
        px.linear_gate_residual(att, w2(5, C), ws[6], c, ws[0], tm, 2 * C, ref)
    elif part == "cross":
        xm = px.layer_norm(ref, 1e-6, ws[7], ws[8], out_dtype=bf)
        q = px.mh_rms_norm(px.linear(xm, w2(9, C), ws[10]), H, 64, ws[13])
        kv = px.linear(ctx, w2(11, 2 * C), ws[12])
        k = px.mh_rms_norm(kv[:, :C].contiguous(), H, 64, ws[14])
        att = px.varlen_attention(q, k, kv[:, C:].contiguous(), cu, off, H, 64, 0.125)
        px.linear_residual(att, w2(15, C), ws[16], ref)
    elif part == "projection":
        px.linear_residual(proj, w2(17, C), ws[18], ref)
    else:
        xm = px.layer_norm_modulate(ref, 1e-6, c, ws[0], tm, 3 * C, out_dtype=bf)
        px.linear_gate_residual(px.linear(xm, w2(19, M), ws[20], act=1), w2(21, C), ws[22], c, ws[0], tm,
                                5 * C, ref)
    err = float((got - ref).norm() / (ref - x).norm())
    print(f"[block bf16 split] relative L2 of the update {err:.2e}", flush=True)
    # sums of K products in other orders, and the update's rounding at the residual's
    # size: a few 2^-24 each
    assert err <= 2e-6
