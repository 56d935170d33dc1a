"""The fp16 prefill form on every tensor type: every number of token tiles and both workgroup forms against the exact-weight product."""
import pytest
import torch

from test_gpu_parity import PLAN_OFFSETS_AT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def half(b):
    return b.contiguous().view(torch.float16).to(torch.float64).squeeze(-1)


def draw(gen, kind, rows, width):
    """Random blocks (every code and factor occurs, small finite fp16 scales) and their values in double precision."""
    per, size, scales = (32, 34, (1,)) if kind == "q8_0" else (256, 176, (1, 3))
    b = torch.randint(0, 256, (rows, width // per, size), dtype=torch.uint8, device="cuda", generator=gen)
    for at in scales:
        b[..., at] = (b[..., at] & 0x03) | 0x0C
    if kind == "q8_0":
        return b.reshape(rows, -1), (half(b[..., 0:2])[..., None] * b[..., 2:].contiguous().view(torch.int8).to(torch.float64)).reshape(rows, width)
    d, dmin, f = half(b[..., 0:2])[..., None], half(b[..., 2:4])[..., None], b[..., 4:16].to(torch.int64)
    out = []
    for j in range(8):                                     # (src/ggml_dequant.cpp: the K-quants' packed six-bit factors)
        sc = f[..., j] & 63 if j < 4 else (f[..., j + 4] & 15) | ((f[..., j - 4] >> 6) << 4)
        mn = f[..., j + 4] & 63 if j < 4 else (f[..., j + 4] >> 4) | ((f[..., j] >> 6) << 4)
        nibbles = b[..., 48 + 32 * (j // 2):80 + 32 * (j // 2)].to(torch.int64)
        q = (nibbles >> 4 if j & 1 else nibbles & 15) | (((b[..., 16:48].to(torch.int64) >> j) & 1) << 4)
        out.append(d * sc[..., None] * q - dmin * mn[..., None])
    return b.reshape(rows, -1), torch.stack(out, -2).reshape(rows, width)


def check_down_product(layer, D, rows, hidden, ffn, experts, top_k, ids):
    """The down rows alone, against double precision on the h that the launch itself read: two fp16 planes, hi and the rest of 22 bits.
    A value takes ffn / 16 matrix operations per plane and a scaled sum per 32 weights, each rounded within 2^-24 of a partial sum, which is no larger
    than the value by rms; the errors' signs are independent, so they add up as the square root of their number, and four times that leaves room
    for the roundings inside an operation. A product without the rest of h, or with a part of it against other weights, is off by more
    than three times the bound (1.2e-5 of the value at ffn 1280 with Q5_K rows throughout, 2e-4 elsewhere), which is checked here as well."""
    pad4 = lambda v: (v + 3) & ~3
    A = rows * top_k
    plane = 2 * (A + 128) * ffn                                                   # bytes of a plane of [assignments in plan order][ffn]
    hi, lo = (layer.h_f16[at:at + 2 * A * ffn].view(torch.float16).reshape(A, ffn).to(torch.float64) for at in (0, plane))
    order_at = PLAN_OFFSETS_AT + pad4(experts + 1) + pad4(experts)
    order = layer.plan[order_at:order_at + A].long()
    expert = ids.reshape(-1).long()[order]
    raw = layer.rawdots.reshape(-1, hidden)[:A].to(torch.float64)[order]
    bound = 4 * 2.0 ** -24 * (2 * (ffn // 16) + ffn // 32) ** 0.5
    off, off_hi, size = 0.0, 0.0, 0.0
    for e in range(experts):
        at, De = (expert == e).nonzero().squeeze(1), D[e * hidden:(e + 1) * hidden]
        want = (hi[at] + lo[at]) @ De.T
        off, off_hi, size = off + float((raw[at] - want).square().sum()), off_hi + float((lo[at] @ De.T).square().sum()), size + float(want.square().sum())
    assert (off / size) ** 0.5 <= bound, ((off / size) ** 0.5, bound)
    assert (off_hi / size) ** 0.5 >= 3 * bound, ((off_hi / size) ** 0.5, bound)


# rows per expert: one tile of 32, two, three and four tiles, an item and a bit, in both workgroup forms; K of an odd number of super-blocks and of one
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(9, 256, 256, 3, 2), (40, 768, 512, 2, 1), (130, 512, 256, 1, 1), (190, 1280, 768, 2, 1), (70, 256, 1280, 1, 1),
                                                           (2100, 512, 512, 32, 2), (2600, 256, 256, 32, 4)])
@pytest.mark.parametrize("gate,down", [("q5_k", "q5_k"), ("q8_0", "q8_0"), ("q5_k", "q8_0"), ("q8_0", "q5_k")])
def test_against_the_exact_product(strix, prefill_form, rows, hidden, ffn, experts, top_k, gate, down):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    (g, G), (u, U), (d, D) = draw(gen, gate, experts * ffn, hidden), draw(gen, gate, experts * ffn, hidden), draw(gen, down, experts * hidden, ffn)
    kinds = dict(gate_type=getattr(strix, "TYPE_" + gate.upper()), down_type=getattr(strix, "TYPE_" + down.upper()))
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows, prefill_f16=True, **kinds)
    x = (torch.randn((rows, hidden), device="cuda", generator=gen) * 0.25).to(torch.float16)
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k, dim=1).indices.to(torch.int32)
    layer.run_prefill_f16(x, ids, torch.rand((rows, top_k), device="cuda", generator=gen))
    prefill_form.check(layer)
    assert int(layer.status[:rows].sum()) == 0
    check_down_product(layer, D, rows, hidden, ffn, experts, top_k, ids)
    raw = layer.rawdots.reshape(-1, hidden)[:rows * top_k].to(torch.float64)
    flat, X = ids.reshape(-1).long(), x.to(torch.float64)
    for e in range(experts):
        at = (flat == e).nonzero().squeeze(1)
        xe, Ge, Ue, De = X[at // top_k], G[e * ffn:(e + 1) * ffn], U[e * ffn:(e + 1) * ffn], D[e * hidden:(e + 1) * hidden]
        a, b = xe @ Ge.T, xe @ Ue.T
        s = 1 / (1 + torch.exp(-a))
        h = a * s * b
        # every product accumulates k / 16 matrix operations and the scaled partial sums of k / 32 blocks in fp32, each within 2^-24 of the sum of
        # magnitudes: no more than (k / 8) 2^-24 of it; the activation's own operations and h's 22 bits add 2^-20 of h
        step = 2.0 ** -24 / 8
        ga, ua = xe.abs() @ Ge.abs().T * (hidden * step), xe.abs() @ Ue.abs().T * (hidden * step)
        slope = (s + a * s * (1 - s)).abs()
        dh = (b.abs() + ua) * slope.clamp(min=0.1) * ga * 1.1 + (a * s).abs() * ua + h.abs() * 2.0 ** -20
        bound = dh @ De.abs().T + h.abs() @ De.abs().T * (ffn * step)
        assert bool(((raw[at] - h @ De.T).abs() <= bound).all()), e


def q4_k_values(b, width):
    """The values of Q4_K blocks in double precision, and the sums of the magnitudes of their two terms."""
    d, dmin, f = half(b[..., 0:2])[..., None], half(b[..., 2:4])[..., None], b[..., 4:16].to(torch.int64)
    out, size = [], []
    for j in range(8):
        sc = f[..., j] & 63 if j < 4 else (f[..., j + 4] & 15) | ((f[..., j - 4] >> 6) << 4)
        mn = f[..., j + 4] & 63 if j < 4 else (f[..., j + 4] >> 4) | ((f[..., j] >> 6) << 4)
        nibbles = b[..., 16 + 32 * (j // 2):48 + 32 * (j // 2)].to(torch.int64)
        scaled, least = d * sc[..., None] * (nibbles >> 4 if j & 1 else nibbles & 15), dmin * mn[..., None]
        out.append(scaled - least)
        size.append(scaled.abs() + least.abs())
    return tuple(torch.stack(v, -2).reshape(-1, width) for v in (out, size))


def draw_q4_k(gen, rows, width):
    """Random blocks; the first weight rows hold the ends of every field: all factors and codes at their largest (sc 63, q 15), no factors, both scales negative,
    a subnormal d, a subnormal dmin."""
    b = torch.randint(0, 256, (rows, width // 256, 144), dtype=torch.uint8, device="cuda", generator=gen)
    for at in (1, 3):
        b[..., at] = (b[..., at] & 0x03) | 0x0C
    b[0, :, 4:] = 0xFF
    b[1, :, 4:16] = 0
    b[2, :, 1] |= 0x80
    b[2, :, 3] |= 0x80
    b[3, :, 0:2] = torch.tensor([0x01, 0x00], dtype=torch.uint8, device="cuda")
    b[4, :, 2:4] = torch.tensor([0xFF, 0x83], dtype=torch.uint8, device="cuda")
    return b


@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(9, 256, 256, 3, 2), (40, 768, 512, 2, 1), (130, 512, 256, 1, 1), (190, 1280, 768, 2, 1), (70, 256, 1280, 1, 1), (600, 512, 512, 8, 2)])
def test_q4_k_against_the_exact_product(strix, prefill_form, rows, hidden, ffn, experts, top_k):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u, d = (draw_q4_k(gen, experts * n, m) for n, m in ((ffn, hidden), (ffn, hidden), (hidden, ffn)))
    (G, Gs), (U, Us), (D, Ds) = q4_k_values(g, hidden), q4_k_values(u, hidden), q4_k_values(d, ffn)
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, *(t.reshape(t.shape[0], -1) for t in (g, u, d)), rows, prefill_f16=True)
    x = (torch.randn((rows, hidden), device="cuda", generator=gen) * 0.25).to(torch.float16)
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k, dim=1).indices.to(torch.int32)
    layer.run_prefill_f16(x, ids, torch.rand((rows, top_k), device="cuda", generator=gen))
    prefill_form.check(layer)
    assert int(layer.status[:rows].sum()) == 0
    check_down_product(layer, D, rows, hidden, ffn, experts, top_k, ids)
    raw = layer.rawdots.reshape(-1, hidden)[:rows * top_k].to(torch.float64)
    flat, X = ids.reshape(-1).long(), x.to(torch.float64)
    # A super-block of a product takes 16 matrix operations a plane (two of h), one for the minimums and two scaled sums in fp32, each within 2^-24 of the
    # terms' magnitudes: 35 at most, here 40. The sums of 32 activations: 31 additions, and 2^-22 as two halves.
    step = lambda k: 2.0 ** -24 * (40 * (k // 256) + 35)
    for e in range(experts):
        at = (flat == e).nonzero().squeeze(1)
        of = lambda t, n: t[e * n:(e + 1) * n]
        xe = X[at // top_k]
        a, b = xe @ of(G, ffn).T, xe @ of(U, ffn).T
        s = 1 / (1 + torch.exp(-a))
        h = a * s * b
        ga, ua = xe.abs() @ of(Gs, ffn).T * step(hidden), xe.abs() @ of(Us, ffn).T * step(hidden)
        slope = (s + a * s * (1 - s)).abs()
        # (the activation's own operations and h's 22 bits: 2^-20 of h; h below fp16's normal range: steps of 2^-24 at most)
        dh = (b.abs() + ua) * slope.clamp(min=0.1) * ga * 1.1 + (a * s).abs() * ua + h.abs() * 2.0 ** -20 + 2.0 ** -24
        bound = (dh + h.abs() * step(ffn)) @ of(Ds, hidden).T
        assert bool(((raw[at] - h @ of(D, hidden).T).abs() <= bound).all()), e


# one infinite or undefined scale or minimum in one gate or up row of an expert: its rows are flagged, the others are not, and nothing is published
@pytest.mark.parametrize("kind", ["q4_k", "q5_k"])
@pytest.mark.parametrize("at,bits", [(0, 0x7C00), (0, 0xFC00), (2, 0x7C00), (2, 0xFC00), (0, 0x7E00)])
def test_scales_that_are_not_finite(strix, prefill_form, kind, at, bits):
    gen = torch.Generator(device="cuda").manual_seed(at + bits)
    rows, hidden, ffn, experts, top_k = 150, 768, 256, 3, 1
    size = {"q4_k": 144, "q5_k": 176}[kind]
    def tensor(n, m):
        b = draw_q4_k(gen, n, m) if kind == "q4_k" else draw(gen, "q5_k", n, m)[0].reshape(n, m // 256, size)
        return b
    g, u, d = tensor(experts * ffn, hidden), tensor(experts * ffn, hidden), tensor(experts * hidden, ffn)
    (g if bits & 0x8000 else u)[ffn + 77, 1, at:at + 2] = torch.tensor([bits & 255, bits >> 8], dtype=torch.uint8, device="cuda")       # of expert 1
    t = getattr(strix, "TYPE_" + kind.upper())
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, *(t_.reshape(t_.shape[0], -1) for t_ in (g, u, d)), rows, prefill_f16=True, gate_type=t, down_type=t)
    x = (torch.randn((rows, hidden), device="cuda", generator=gen) * 0.25).to(torch.float16)
    ids = torch.randint(0, experts, (rows, 1), device="cuda", generator=gen).to(torch.int32)
    layer.output.fill_(-7.0)
    y = layer.run_prefill_f16(x, ids, torch.ones((rows, 1), device="cuda"))
    prefill_form.check(layer)
    assert torch.equal(layer.status[:rows] & strix.STATUS_NONFINITE_PROJECTION != 0, ids[:, 0] == 1) and bool((y == -7.0).all())
