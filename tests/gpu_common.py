"""Shared helpers for the GPU parity tests (they call libpxs.so through pxs.py)."""

import numpy as np
import torch

FP32_TOL = 1e-5   # max|g - r| / max|r|
BF16_TOL = 1e-2   # relative L2


def dev():
    return torch.device("cuda:0")


def t32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev())


def ti32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(dev())


def ti64(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int64)).to(dev())


def tbf(a):
    """float32 numpy (already bf16-representable or not) -> bf16 device tensor (RNE)."""
    return t32(a).to(torch.bfloat16)


def host(t):
    return t.detach().float().cpu().numpy()


def random_flow(dtype, channels, blocks, latent, seed):
    """A SLat-flow model with random weights on the device -> (FlowConfig,
    FlowWeights, the list of its blocks' tensors, what has to be kept alive)."""
    import pxs
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s, std=1.0: torch.randn(*s, device="cuda", generator=gen) * std  # noqa: E731
    ch = channels
    cfg = pxs.FlowConfig(latent, latent, ch, ch, blocks, ch // 64, 0, 4 * ch, 1e-6, 1.0, 10000.0, 1, 1, 0)
    fw = [rand(ch, latent, std=0.2), rand(ch), rand(ch, 256, std=0.02), rand(ch), rand(ch, ch, std=0.02),
          rand(ch), rand(6 * ch, ch, std=0.02), rand(6 * ch, std=0.1), rand(latent, ch, std=0.03),
          rand(latent)]
    sizes = [6 * ch, 3 * ch * ch, 3 * ch, ch, ch, ch * ch, ch, ch, ch, ch * ch, ch, 2 * ch * ch, 2 * ch,
             ch, ch, ch * ch, ch, 0, 0, 4 * ch * ch, 4 * ch, 4 * ch * ch, ch]
    tensors = []
    for _ in range(blocks):
        ws = [rand(n, std=0.03) if n else None for n in sizes]
        for i in (3, 4, 7, 13, 14):  # RMS gammas and the norm2 weight
            ws[i] = ws[i] + 1.0
        tensors.append([w.to(dtype) if w is not None and i in pxs.BLOCK_LINEAR_WEIGHTS else w
                        for i, w in enumerate(ws)])
    arr = (pxs.BlockWeights * blocks)(*[pxs.block_weights(b) for b in tensors])
    return cfg, pxs.FlowWeights(*[a.data_ptr() for a in fw], arr), tensors, (fw, arr)


def max_rel(got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    denom = max(float(np.max(np.abs(ref))), 1e-30)
    return float(np.max(np.abs(got - ref))) / denom


def rel_l2(got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    return float(np.linalg.norm(got - ref) / max(np.linalg.norm(ref), 1e-30))


def assert_fp32(got, ref, tol=FP32_TOL, what=""):
    e = max_rel(got, ref)
    assert e <= tol, f"{what}: max rel error {e:.3e} > {tol}"


def assert_bf16(got, ref, tol=BF16_TOL, what=""):
    e = rel_l2(got, ref)
    assert e <= tol, f"{what}: rel L2 error {e:.3e} > {tol}"
