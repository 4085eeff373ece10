"""Workspace sizes (host functions of libpxs.so, no GPU): each query covers
every layout that the call it sizes can carve."""

import ctypes as C

import pytest

import pxs

LIB = pxs.load_library()


def up(nbytes):
    return (nbytes + 255) // 256 * 256  # each buffer is 256-byte aligned


def flow_config(channels, heads, blocks, cond_channels, latent=32, mlp_ratio=4):
    return pxs.FlowConfig(latent, latent, channels, cond_channels, blocks, heads, 0,
                          mlp_ratio * channels, 1e-6, 1.0, 10000.0, 1, 1, 0)


def flow_bytes(dtype, cfg, rows, tokens, batch):
    return LIB.pxs_slat_flow_workspace_bytes(dtype, C.byref(cfg), rows, tokens, batch)


def sampler_bytes(dtype, cfg, rows, cond, uncond, batch):
    return LIB.pxs_flow_euler_sample_workspace_bytes(dtype, C.byref(cfg), rows, cond, uncond, batch)


@pytest.mark.parametrize("dtype", [pxs.PXS_BF16, pxs.PXS_F32])
@pytest.mark.parametrize("channels,heads,blocks", [(1024, 16, 24), (1536, 24, 30), (256, 4, 2)])
@pytest.mark.parametrize("cond,uncond", [(1370, 1370), (5000, 1), (1, 9000), (2621, 2622)])
def test_sampler_workspace_holds_every_step(dtype, channels, heads, blocks, cond, uncond):
    """A guided step runs the forward over twice the rows, an unguided one over
    the rows alone with either context, all in the workspace's last buffer."""
    cfg = flow_config(channels, heads, blocks, 1024)
    e = 2 if dtype == pxs.PXS_BF16 else 4
    for batch in (1, 3):
        for rows in (3, 700, 1344, 1345, 2688, 2689, 4095, 4096, 4097, 4600, 5000, 8192, 8193):
            front = (up(2 * rows * 16) + 2 * up((2 * batch + 1) * 8) + up(2 * rows * 32 * 4) +
                     up(2 * batch * 4) + up((cond + uncond) * 1024 * e) + up(2 * rows * 32 * 4) +
                     2 * up(rows * 32 * 4) + up(8) +
                     up(LIB.pxs_flow_guidance_workspace_bytes(batch)))
            have = sampler_bytes(dtype, cfg, rows, cond, uncond, batch) - front
            for r, tokens, b in ((2 * rows, cond + uncond, 2 * batch), (rows, cond, batch),
                                 (rows, uncond, batch)):
                need = flow_bytes(dtype, cfg, r, tokens, b)
                assert need <= have, (f"rows {rows}, batch {batch}: a step over {r} rows and {tokens} "
                                      f"tokens uses {need} of {have} bytes")


def never_shrinks(sizes, what):
    worst = max(zip(sizes, sizes[1:]), key=lambda p: p[0] - p[1])
    assert worst[0] <= worst[1], f"{what}: {worst[0]} bytes, then {worst[1]} for a larger call"


ROWS = sorted({1, 7, 100, *(k + d for k in (128, 1344, 1664, 2688, 3328, 4096, 6656, 10880, 8192, 10752, 21760, 43520)
                            for d in (-1, 0, 1))})


@pytest.mark.parametrize("dtype", [pxs.PXS_BF16, pxs.PXS_F32])
@pytest.mark.parametrize("channels,heads,blocks", [(1024, 16, 24), (1536, 24, 30), (256, 4, 2)])
def test_flow_and_block_workspaces_serve_every_smaller_call(dtype, channels, heads, blocks):
    """One workspace of the largest call's size serves calls of fewer rows,
    context tokens and items: the sizes never fall as any of them grows."""
    cfg = flow_config(channels, heads, blocks, 1024)
    block = pxs.BlockConfig(channels, heads, 4 * channels, 1024, 512, 1e-6, 1.0, 10000.0, 1, 1, 1, 1)
    cap = (1 << 29) // (4 * channels * blocks)  # tokens whose keys and values of all blocks are 512 MB
    tokens = sorted({0, 1, 1370, cap - 1, cap, cap + 1, 2 * cap, 40000})
    sizes = {
        "flow": lambda r, t, b: flow_bytes(dtype, cfg, r, t, b),
        "block": lambda r, t, b: LIB.pxs_transformer_block_workspace_bytes(dtype, C.byref(block), r, t, b),
        "sampler": lambda r, t, b: sampler_bytes(dtype, cfg, r, t, t, b),
    }
    for name, size in sizes.items():
        for b in (1, 2, 5):
            for t in tokens:
                never_shrinks([size(r, t, b) for r in ROWS], f"{name}, {t} tokens, growing rows")
            for r in ROWS:
                never_shrinks([size(r, t, b) for t in tokens], f"{name}, {r} rows, growing tokens")
        never_shrinks([size(3000, 1370, b) for b in range(1, 70)], f"{name}, growing items")


def test_decoder_workspaces_serve_every_smaller_call():
    for dtype in (pxs.PXS_BF16, pxs.PXS_F32):
        for ch in (64, 256, 1024):
            never_shrinks([LIB.pxs_convnext_block_workspace_bytes(dtype, r, ch, 4 * ch, 1) for r in ROWS],
                          "ConvNeXt block, growing rows")
            never_shrinks([LIB.pxs_resblock_c2s_workspace_bytes(dtype, r, ch, ch // 2) for r in ROWS],
                          "up-block, growing rows")


def test_sizes_of_refused_configurations():
    """A size query answers for configurations that the call then refuses."""
    for ch in (0, -256):
        cfg = flow_config(ch, 4, 2, 64)
        block = pxs.BlockConfig(ch, 4, 256, 64, 0, 1e-6, 1.0, 10000.0, 1, 1, 1, 0)
        for dtype in (pxs.PXS_BF16, pxs.PXS_F32):
            for rows in (0, 100):
                flow_bytes(dtype, cfg, rows, 10, 1)
                LIB.pxs_transformer_block_workspace_bytes(dtype, C.byref(block), rows, 10, 1)
    assert LIB.pxs_slat_flow_workspace_bytes(pxs.PXS_BF16, None, 100, 10, 1) == 0
    assert LIB.pxs_transformer_block_workspace_bytes(pxs.PXS_BF16, None, 100, 10, 1) == 0
