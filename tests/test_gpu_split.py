"""fp32 products on the bf16 matrix cores (csrc/split3.h): operands split into
three bf16 terms, six of nine products.

* Products with one: every operand comes back bit for bit, which takes each of
  the three planes of either operand.
* Sums against 64 bits: relative 2-norms that a split without its third plane
  does not reach (computed here on the CPU).
* Operands at the edge of the split's range: below 2^-110 they lose bits, so a
  sum that this could move by more than fp32's own rounding is taken again on
  the fp32 instruction, and one that it cannot is not.
* An output depends on its own row and channel only, whatever its tile holds."""

import numpy as np
import pytest
import torch

import pxs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def px():
    return pxs.Pxs()


def gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def mantissas(g, *shape):
    """Random signs and full 24-bit mantissas over exponents -20 .. 20."""
    m = 1 + torch.randint(0, 1 << 23, shape, generator=g, device="cuda").double() * 2.0 ** -23
    s = 1 - 2 * torch.randint(0, 2, shape, generator=g, device="cuda")
    e = torch.randint(-20, 21, shape, generator=g, device="cuda")
    return (m * s * torch.exp2(e.double())).float()


def slab(rows):
    """Coordinates of a two-voxel-thick plate, 200 rows per x."""
    i = torch.arange(rows, device="cuda")
    return torch.stack([0 * i, i // 200, i // 2 % 100, i % 2], 1).to(torch.int32)


def conv64(x, w, nbr, rows):
    """The convolution's sums at some rows in 64 bits."""
    n = x.shape[0]
    ref = torch.zeros(rows.shape[0], w.shape[1], dtype=torch.float64, device=x.device)
    for k in range(27):
        src = nbr[k][rows].long()
        ref[src != n] += x[src[src != n]].double() @ w[k].double().t()
    return ref


def attn64(q, k, v, heads, scale):
    out = torch.empty(q.shape[0], heads * 64, dtype=torch.float64, device=q.device)
    for h in range(heads):
        c = slice(64 * h, 64 * h + 64)
        s = q[:, c].double() @ k[:, c].double().t().contiguous() * scale
        out[:, c] = torch.softmax(s, 1) @ v[:, c].double()
    return out


def bounds(*lens):
    return torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device="cuda")


def rel(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


# The three tile shapes of the linear, its K splits' grid apart.
LINEAR_ROWS = [(40, 64), (3000, 64), (20000, 64), (9000, 256)]


@pytest.mark.parametrize("rows,k", LINEAR_ROWS)
def test_linear_times_one_is_exact(px, rows, k):
    g = gen(rows)
    x, eye = mantissas(g, rows, k), torch.eye(k, device="cuda")
    w = mantissas(g, 132, k)
    ones = eye.repeat(rows // k + 1, 1)[:rows].contiguous()
    print(f"[split linear] {rows} x {k}", flush=True)
    assert torch.equal(px.linear(x, eye), x)
    assert torch.equal(px.linear(ones, w), w.t().repeat(rows // k + 1, 1)[:rows])


def test_conv_times_one_is_exact(px):
    n, c = 17000, 64
    g = gen(1)
    coords = slab(n)
    nbr, masks = px.neighbor_map(coords)
    x, w = mantissas(g, n, c), torch.zeros(27, c, c, device="cuda")
    w[13] = torch.eye(c, device="cuda")
    print(f"[split conv] {n} rows", flush=True)
    assert torch.equal(px.subm_conv3d(x, w, None, nbr, masks), x)
    w[13] = mantissas(g, c, c)
    ones = torch.eye(c, device="cuda").repeat(n // c + 1, 1)[:n].contiguous()
    assert torch.equal(px.subm_conv3d(ones, w, None, nbr, masks), w[13].t().repeat(n // c + 1, 1)[:n])


def test_attention_of_one_key_is_exact(px):
    """A segment of one key: its value, all three planes of it."""
    g = gen(2)
    heads, nseg, lens = 16, 8, [300] * 8
    q, k, v = normal(g, sum(lens), 64 * heads), normal(g, nseg, 64 * heads), mantissas(g, nseg, 64 * heads)
    v[1] *= 2.0 ** -120  # subnormals among them
    v[2] = 2.0 ** -140
    v[3, ::2] = 0.0
    print("[split attention] one key", flush=True)
    o = px.varlen_attention(q, k, v, bounds(*lens), bounds(*[1] * nseg), heads, 64, 0.125)
    assert torch.equal(o, v.repeat_interleave(300, 0))


def two_planes(a):
    """a rounded to its first two bf16 terms."""
    hi = a.to(torch.bfloat16).float()
    return hi + (a - hi).to(torch.bfloat16).float()


# Bounds: twice what was measured (1.1e-7, 4.9e-7, 1.0e-6 at K = 64, 1024 and 4096)
# and more; two planes of one operand give 2.4e-6.
@pytest.mark.parametrize("rows,k,n,bound", [(3000, 64, 260, 4e-7), (3000, 1024, 520, 1e-6),
                                            (1000, 4096, 260, 2e-6)])
def test_linear_sums(px, rows, k, n, bound):
    g = gen(rows + k)
    x, w = normal(g, rows, k), normal(g, n, k)
    ref = x.double() @ w.double().t()
    err = rel(px.linear(x, w), ref)
    print(f"[split linear] {rows}x{k}->{n} relative L2 {err:.2e}", flush=True)
    assert err <= bound
    s = slice(0, 200)
    planted = rel(two_planes(x[s].cpu()).double() @ w.cpu().double().t(), ref[s].cpu())
    print(f"[split linear] two planes {planted:.2e}", flush=True)
    assert planted > bound


@pytest.mark.parametrize("cin,cout,bound", [(4, 130, 5e-7), (36, 192, 5e-7), (128, 129, 5e-7)])
def test_conv_sums(px, cin, cout, bound):
    n = 17000
    g = gen(cin)
    nbr, masks = px.neighbor_map(slab(n))
    x, w = normal(g, n, cin), normal(g, 27, cout, cin)
    rows = torch.arange(0, n, 13, device="cuda")
    ref = conv64(x, w, nbr, rows)
    err = rel(px.subm_conv3d(x, w, None, nbr, masks)[rows], ref)
    print(f"[split conv] {cin}->{cout} relative L2 {err:.2e}", flush=True)
    assert err <= bound
    planted = rel(conv64(two_planes(x.cpu()), w.cpu(), nbr.cpu(), rows.cpu()), ref.cpu())
    print(f"[split conv] two planes {planted:.2e}", flush=True)
    assert planted > bound


@pytest.mark.parametrize("heads,n,gain,bound", [(16, 1100, 1.0, 1.1e-6), (16, 1100, 6.0, 1.7e-6)])
def test_attention_sums(px, heads, n, gain, bound):
    g = gen(int(gain))
    q, k, v = (normal(g, n, 64 * heads) for _ in range(3))
    q = q * gain
    ref = attn64(q, k, v, heads, 0.125)
    err = rel(px.varlen_attention(q, k, v, bounds(n), bounds(n), heads, 64, 0.125), ref)
    print(f"[split attention] gain {gain} relative L2 {err:.2e}", flush=True)
    assert err <= bound
    c = [t[:, :64].cpu() for t in (q, k, v)]
    for i in range(3):  # one operand without its third plane
        planted = rel(attn64(*[two_planes(t) if j == i else t for j, t in enumerate(c)], 1, 0.125),
                      ref[:, :64].cpu())
        print(f"[split attention] two planes of operand {i}: {planted:.2e}", flush=True)
        assert planted > bound


def test_linear_of_small_operands_keeps_their_bits(px):
    """Every x is 2^-119 (1 + 2^-15), whose last bit is half the least step of a
    bf16 plane, every w 2^50, the largest operand the split takes: without that
    bit the sum is off by 2^-15 of itself.  With it, up to 256 equal terms add up
    without rounding in fp32; 1,024 round to 2^-16 (their sums' last bit)."""
    for k in (64, 256, 1024):
        x = torch.full((300, k), (1 + 2.0 ** -15) * 2.0 ** -119, device="cuda")
        w = torch.full((130, k), 2.0 ** 50, device="cuda")
        ref = k * (1 + 2.0 ** -15) * 2.0 ** -69
        for y in (px.linear(x, w), px.linear(w, x)):
            err = (y.double() - ref).abs().max().item() / ref
            print(f"[split range] K {k} small operands: {err:.2e}", flush=True)
            assert err <= (2.0 ** -16 if k == 1024 else 0.0)


# x at 2^e, w at 2^f, K terms of one sign: (-121, 49): the sums are above 2^-60, and
# the operands keep 12 bits of 24; (-108, 49): every bit kept; (-83, 0): ordinary
# weights and tiny features; (-130, 20), (-140, 0): subnormals, the latter below the
# least term a bf16 plane holds.
RANGES = [(-121, 49, 4096), (-112, 49, 1024), (-108, 49, 256), (-83, 0, 512), (-100, -5, 64),
          (-130, 20, 64), (-140, 0, 64), (20, -140, 64), (-60, -66, 64)]


@pytest.mark.parametrize("e,f,k", RANGES)
def test_linear_edges_of_range(px, e, f, k):
    g = gen(1000 - e + f)
    x = (1 + torch.rand(300, k, generator=g, device="cuda").double()) * 2.0 ** e
    w = (1 + torch.rand(130, k, generator=g, device="cuda").double()) * 2.0 ** f
    x, w = x.float(), w.float()  # subnormals rounded to what fp32 holds
    ref = x.double() @ w.double().t()
    y = px.linear(x, w).double()
    # K fp32 additions of one sign, and the least step of subnormal products and sums
    room = ref * k * 2.0 ** -24 + k * 2.0 ** -149
    worst = ((y - ref).abs() / room).max().item()
    print(f"[split range] linear 2^{e} x 2^{f}, K {k}: error / room {worst:.2e}", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("e,f", [(e, f) for e, f, k in RANGES])
def test_conv_edges_of_range(px, e, f):
    n, cin, cout = 17000, 32, 64
    g = gen(2000 - e + f)
    nbr, masks = px.neighbor_map(slab(n))
    x = ((1 + torch.rand(n, cin, generator=g, device="cuda").double()) * 2.0 ** e).float()
    w = ((1 + torch.rand(27, cout, cin, generator=g, device="cuda").double()) * 2.0 ** f).float()
    rows = torch.arange(0, n, 13, device="cuda")
    ref = conv64(x, w, nbr, rows)
    y = px.subm_conv3d(x, w, None, nbr, masks)[rows].double()
    worst = ((y - ref).abs() / (ref * 27 * cin * 2.0 ** -24 + 27 * cin * 2.0 ** -149)).max().item()
    print(f"[split range] conv 2^{e} x 2^{f}: error / room {worst:.2e}", flush=True)
    assert worst <= 1.0


# Values at 2^e beside a query at 2^f (which sets the largest operand), and
# scores from tiny queries under a large scale.
@pytest.mark.parametrize("e,f,qe,scale", [(-83, 0, 0, 0.125), (-121, 40, 0, 0.125), (-130, 0, 0, 0.125),
                                          (0, 0, -112, 2.0 ** 108),
                                          (0, 0, -70, 2.0 ** 68)])
def test_attention_edges_of_range(px, e, f, qe, scale):
    heads, n = 16, 1100
    g = gen(3000 - e + f)
    q, k = normal(g, n, 64 * heads) * 2.0 ** qe, normal(g, n, 64 * heads)
    v = ((1 + torch.rand(n, 64 * heads, generator=g, device="cuda").double()) * 2.0 ** e).float()
    q[5], k[:, 0] = q[5] * 0, 0.0
    q[5, 0] = 2.0 ** f if f else 0.0  # the key is 0 there
    ref = attn64(q, k, v, heads, scale)
    o = px.varlen_attention(q, k, v, bounds(n), bounds(n), heads, 64, scale).double()
    worst = ((o - ref).abs() / (ref * 2.0 ** -18 + 4 * n * 2.0 ** -149)).max().item()
    print(f"[split range] attention v 2^{e} q[5] 2^{f} q 2^{qe} scale {scale:g}: error / room {worst:.2e}",
          flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("what", ["inf", "nan", "huge", "tiny", "zero"])
def test_linear_rows_do_not_touch_each_other(px, what):
    """One row out of range: the others' bits are those of a call without it."""
    g = gen(77)
    x, w = normal(g, 1000, 256), normal(g, 200, 256)
    y = px.linear(x, w)
    x2 = x.clone()
    x2[333] = {"inf": torch.inf, "nan": torch.nan, "huge": 1e25, "tiny": 1e-35, "zero": 0.0}[what]
    y2 = px.linear(x2, w)
    keep = torch.arange(1000, device="cuda") != 333
    assert torch.equal(y2[keep], y[keep])
    ref = x2[333].double() @ w.double().t()
    assert torch.equal(torch.isnan(y2[333]), torch.isnan(ref))
    if what in ("huge", "tiny", "zero"):
        assert ((y2[333] - ref).abs() <= 256 * 2.0 ** -24 * (x2[333].double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("what", ["inf", "huge", "tiny"])
def test_conv_rows_do_not_touch_each_other(px, what):
    n, c = 17000, 64
    g = gen(78)
    nbr, masks = px.neighbor_map(slab(n))
    x, w = normal(g, n, c), normal(g, 27, c, c)
    y = px.subm_conv3d(x, w, None, nbr, masks)
    x2 = x.clone()
    x2[5000] = {"inf": torch.inf, "huge": 1e25, "tiny": 1e-35}[what]
    y2 = px.subm_conv3d(x2, w, None, nbr, masks)
    far = ~(nbr == 5000).any(0)
    assert torch.equal(y2[far], y[far])


# Zeros of zero rows, of zero channels, of both, and of operands so small that no
# plane holds them; few zero rows (looked through by row) and few zero channels.
@pytest.mark.parametrize("rows,k,n", [(700, 64, 130), (3000, 512, 260), (200, 36, 68)])
@pytest.mark.parametrize("zero_rows,zero_channels", [(3, 0), (0, 3), (2, 2), (97, 1)])
@pytest.mark.parametrize("tiny", [False, True])
def test_linear_zeros(px, rows, k, n, zero_rows, zero_channels, tiny):
    g = gen(rows + zero_rows)
    x, w = normal(g, rows, k), normal(g, n, k)
    if zero_rows:
        x[::zero_rows + 7] = 0.0
    if zero_channels:
        w[::zero_channels + 5] = 0.0
    if tiny:
        x[11::50] = 2.0 ** -140
        x[12::50] *= 2.0 ** -142
        w[7::40] *= 2.0 ** -141
    print(f"[split zeros] {rows}x{k}->{n} zero rows {zero_rows} channels {zero_channels} tiny {tiny}", flush=True)
    y = px.linear(x, w).double()
    ref = x.double() @ w.double().t()
    room = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + k * 2.0 ** -149
    assert ((y - ref).abs() <= room).all()
    assert (y[(x == 0).all(1)] == 0).all() and (y[:, (w == 0).all(1)] == 0).all()
    if tiny:  # fp32 keeps them
        assert (y[11::50].abs().sum(1) > 0).all()


@pytest.mark.parametrize("tiny", [False, True])
def test_conv_zeros(px, tiny):
    n, c = 17000, 64
    g = gen(5)
    nbr, masks = px.neighbor_map(slab(n))
    x, w = normal(g, n, c), normal(g, 27, c, c)
    x[2000:6000] = 0.0
    w[:, 9] = 0.0
    if tiny:
        x[3000:3400] = 2.0 ** -140
    print(f"[split zeros] conv tiny {tiny}", flush=True)
    y = px.subm_conv3d(x, w, None, nbr, masks).double()
    rows = torch.arange(1500, 6500, 3, device="cuda")
    ref, room = conv64(x, w, nbr, rows), conv64(x.abs(), w.abs(), nbr, rows)
    assert ((y[rows] - ref).abs() <= 27 * c * (2.0 ** -24 * room + 2.0 ** -149)).all()
    assert (y[:, 9] == 0).all() and (y[2600:2790] == 0).all()
    if tiny:
        assert (y[3200].abs().sum() > 0).item()
