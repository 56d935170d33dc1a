"""Decode layers planned from early routes with Q6_K, Q8_0 or Q5_1 down rows: the bits of the staged launches on the exact router's choice."""
import pytest
import torch

import orc
from test_gpu_parity import early_choice

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def blocks(gen, rows, width, per, size, scales):
    w = torch.randint(0, 256, (rows, width // per, size), dtype=torch.uint8, device="cuda", generator=gen)
    for at in scales:
        w[..., at] = (w[..., at] & 0x03) | 0x0C
    return w.reshape(rows, -1)


# the word of the plan that the down launch of a layer with early routes, and no other, moves on by one
EPOCH = 672 + 3 * 16 * 32 + 16


# eight assignments (the fewest of this form) up to 128 (the most); rows of one and of several stages
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k,amount", [(1, 2048, 768, 128, 8, 40), (16, 1024, 512, 32, 8, 40), (7, 512, 256, 24, 5, 300), (4, 768, 1280, 16, 2, 0)])
@pytest.mark.parametrize("down", ["q6_k", "q8_0", "q5_1"])
def test_early_routes_equal_staged_launches(strix, rows, hidden, ffn, experts, top_k, amount, down):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u = (blocks(gen, experts * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, experts * hidden, ffn, *{"q6_k": (256, 210, (209,)), "q8_0": (32, 34, (1,)), "q5_1": (32, 24, (1, 3))}[down])
    layer, staged = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows, down_type=getattr(strix, "TYPE_" + down.upper())) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)
    base = torch.randn((rows, hidden), device="cuda", generator=gen)
    ids, w = strix.route(x, router, top_k)[:2]

    if amount:                     # the displaced early choice is another one in some slots
        assert int((torch.from_numpy(early_choice(x.cpu().numpy(), router.cpu().numpy(), top_k, amount).astype("int64")) != ids.cpu()).sum()) >= 2

    def run(displaced, form, b):
        epoch = int(layer.plan[EPOCH])
        strix.lib().mi355_debug_early_route_perturb(displaced)
        try:
            y, got, weights, _ = layer.run_layer(x, router, base=b, combine=form)
            torch.cuda.synchronize()
            assert int(layer.plan[EPOCH]) == epoch + 1
        finally:
            strix.lib().mi355_debug_early_route_perturb(0)
        assert int(layer.status[:rows].sum()) == 0 and torch.equal(got, ids) and torch.equal(weights.view(torch.int32), w.view(torch.int32))
        return y.clone()

    for form in (strix.COMBINE_FMA_SLOT, strix.COMBINE_MULADD_ASC):
        for b in (None, base):
            want = staged.run(x, ids, w, base=b, combine=form)
            for displaced in (0, amount):
                assert torch.equal(run(displaced, form, b).view(torch.int32), want.view(torch.int32)), (form, displaced)
    # a row whose projection overflows: the same status as the staged launches give, no row published, and the next call is whole again
    good, x0 = run(0, strix.COMBINE_FMA_SLOT, None), x.clone()
    wide = x.to(torch.float32)
    wide[rows - 1] *= 1e37
    layer.output.fill_(7.0)
    y, got, weights, _ = layer.run_layer(wide, router)
    staged.run(wide, got.clone(), weights.clone())
    assert torch.equal(layer.status[:rows], staged.status[:rows]) and int(layer.status[rows - 1]) != 0
    assert bool((layer.output[:rows] == 7.0).all())
    x.copy_(x0)
    assert torch.equal(run(amount, strix.COMBINE_FMA_SLOT, None).view(torch.int32), good.view(torch.int32))


# fp32 rows, whose exact chain holds the row in registers (one step of 16 features each), and rows normalised in front of the launch
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(2, 256, 256, 16, 4), (16, 1280, 256, 24, 8), (9, 2048, 512, 48, 4)])
@pytest.mark.parametrize("norm", [None, torch.float32, torch.bfloat16])
def test_fp32_rows_equal_staged_launches(strix, rows, hidden, ffn, experts, top_k, norm):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u = (blocks(gen, experts * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, experts * hidden, ffn, 256, 210, (209,))
    layer, staged = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows, down_type=strix.TYPE_Q6_K) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(norm or torch.float32)
    scale = torch.rand((hidden,), device="cuda", generator=gen)
    for displaced in (0, 60):
        epoch = int(layer.plan[EPOCH])
        strix.lib().mi355_debug_early_route_perturb(displaced)
        try:
            y, ids, w, scores = layer.run_layer(x, router, norm=(scale, 1e-6) if norm else None)
            torch.cuda.synchronize()
            assert int(layer.plan[EPOCH]) == epoch + 1
        finally:
            strix.lib().mi355_debug_early_route_perturb(0)
        rows32 = strix.rmsnorm_f32(x.to(torch.float32), scale, 1e-6) if norm else x
        if norm:
            assert torch.equal(layer.normed[:rows].view(torch.int32), rows32.view(torch.int32))
        want_ids, want_w, want_scores = strix.route(rows32, router, top_k)
        if displaced:
            assert int((torch.from_numpy(early_choice(rows32.cpu().numpy(), router.cpu().numpy(), top_k, displaced).astype("int64")) != want_ids.cpu()).sum()) >= 2
        assert torch.equal(ids, want_ids) and torch.equal(w.view(torch.int32), want_w.view(torch.int32))
        assert torch.equal(scores.reshape(-1)[:rows * experts].view(torch.int32), want_scores.reshape(-1).view(torch.int32))
        assert torch.equal(y.view(torch.int32), staged.run(rows32, want_ids, want_w).view(torch.int32)) and int(layer.status[:rows].sum()) == 0


# rows of more chunks than the side chain's ring has places, the last one partial; more rows than two rounds of the down + combine launch; sweeps of whole and of
# partial stages; images of h that a repair copies in one piece and in several
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(1, 2304, 256, 16, 8), (3, 3328, 256, 24, 4), (16, 4096, 256, 16, 8), (5, 4096, 2304, 10, 8), (2, 8192, 256, 24, 16),
                                                           (10, 4096, 512, 16, 8), (11, 4096, 512, 16, 8), (6, 8192, 2048, 10, 8)])
@pytest.mark.parametrize("dtype,down", [(torch.float16, "q4_k"), (torch.bfloat16, "q8_0"), (torch.float32, "q4_k")])
def test_long_rows_equal_staged_launches(strix, rows, hidden, ffn, experts, top_k, dtype, down):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u = (blocks(gen, experts * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, experts * hidden, ffn, *{"q4_k": (256, 144, (1, 3)), "q8_0": (32, 34, (1,))}[down])
    layer, staged = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows, down_type=getattr(strix, "TYPE_" + down.upper())) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(dtype)
    ids, w, scores = (t.clone() for t in strix.route(x, router, top_k))
    want = staged.run(x, ids, w)
    assert int((torch.from_numpy(early_choice(x.float().cpu().numpy(), router.cpu().numpy(), top_k, 150).astype("int64")) != ids.cpu()).sum()) >= 2
    for displaced in (0, 150, 0):
        epoch = int(layer.plan[EPOCH])
        strix.lib().mi355_debug_early_route_perturb(displaced)
        try:
            y, got, weights, s = layer.run_layer(x, router)
            torch.cuda.synchronize()
        finally:
            strix.lib().mi355_debug_early_route_perturb(0)
        assert int(layer.plan[EPOCH]) == epoch + 1 and int(layer.status[:rows].sum()) == 0
        assert torch.equal(got, ids) and torch.equal(weights.view(torch.int32), w.view(torch.int32))
        assert torch.equal(s.reshape(-1)[:rows * experts].view(torch.int32), scores.reshape(-1).view(torch.int32))
        assert torch.equal(y.view(torch.int32), want.view(torch.int32)), displaced


# always-on slots: nine (an instance of their own), ten and more, up to eight; with and without a gate; as many assignments as the form takes
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k,shared", [(1, 2048, 256, 24, 8, 1), (14, 1792, 256, 32, 8, 1), (5, 2048, 768, 16, 6, 2), (8, 2304, 256, 24, 14, 2), (6, 1792, 512, 16, 8, 2),
                                                                  (2, 256, 256, 16, 4, 1), (14, 1280, 1024, 16, 8, 1), (4, 1536, 1536, 12, 4, 2)])
@pytest.mark.parametrize("down", ["q4_k", "q6_k", "q8_0", "q5_1"])
@pytest.mark.parametrize("gated", [False, True])
def test_always_on_slots_equal_the_router_launch(strix, rows, hidden, ffn, experts, top_k, shared, down, gated):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + top_k)
    E, K = experts + shared, top_k + shared
    g, u = (blocks(gen, E * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, E * hidden, ffn, *{"q4_k": (256, 144, (1, 3)), "q6_k": (256, 210, (209,)), "q8_0": (32, 34, (1,)), "q5_1": (32, 24, (1, 3))}[down])
    layer, staged = (strix.MoeLayer(hidden, ffn, E, K, g, u, d, rows, down_type=getattr(strix, "TYPE_" + down.upper())) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)
    gates = torch.rand((rows, shared), device="cuda", generator=gen) if gated else None
    ids, w = (t.clone() for t in strix.route(x, router, top_k)[:2])
    all_ids = torch.cat([ids, torch.arange(experts, E, device="cuda", dtype=torch.int32).expand(rows, shared)], dim=1).contiguous()
    all_w = torch.cat([w, gates if gated else torch.ones((rows, shared), device="cuda")], dim=1).contiguous()
    staged.run(x, all_ids, all_w)
    for form in (strix.COMBINE_FMA_SLOT, strix.COMBINE_MULADD_ASC):
        want = orc.combine_shared(form, all_w.cpu().numpy(), all_ids.cpu().numpy(), staged.rawdots[:rows].cpu().numpy().reshape(rows, K, hidden), shared)
        for displaced in (0, 200):
            epoch = int(layer.plan[EPOCH])
            strix.lib().mi355_debug_early_route_perturb(displaced)
            try:
                y, got, weights, _ = layer.run_layer(x, router, combine=form, shared_experts=shared, shared_slot_weights=gates)
                torch.cuda.synchronize()
            finally:
                strix.lib().mi355_debug_early_route_perturb(0)
            assert int(layer.plan[EPOCH]) == epoch + 1 and int(layer.status[:rows].sum()) == 0
            assert torch.equal(got, all_ids) and torch.equal(weights.view(torch.int32), all_w.view(torch.int32))
            assert torch.equal(layer.rawdots[:rows].view(torch.int32), staged.rawdots[:rows].view(torch.int32))
            assert torch.equal(y.view(torch.int32), torch.from_numpy(want).cuda().view(torch.int32)), (form, displaced)


# the lines up to which always-on experts take early routes: of their bytes (9 | 10 rows of 1792 / 2048, 4 | 5 of 3072 / 2304), the experts' width and the slots of
# rows of up to 1536 features; a row's bits are the same on both sides
@pytest.mark.parametrize("hidden,ffn,top_k,early,late", [(1792, 2048, 4, 9, 10), (3072, 2304, 4, 5, 6), (1280, 1280, 4, 5, None), (1280, 1536, 4, None, 5), (1024, 256, 3, None, 16)])
@pytest.mark.parametrize("norm", [False, True])
def test_lines_of_always_on_experts(strix, hidden, ffn, top_k, early, late, norm):
    gen = torch.Generator(device="cuda").manual_seed(hidden + ffn)
    experts, rows = 16, max(early or 0, late or 0)
    g, u = (blocks(gen, (experts + 1) * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, (experts + 1) * hidden, ffn, 256, 144, (1, 3))
    layer = strix.MoeLayer(hidden, ffn, experts + 1, top_k + 1, g, u, d, rows)
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)
    scale = torch.rand((hidden,), device="cuda", generator=gen)
    singles = [layer.run_layer(x[i:i + 1], router, shared_experts=1, norm=(scale, 1e-6) if norm else None)[0].clone() for i in range(rows)]
    for n, moved in ((early, 1), (late, 0)):
        if not n:
            continue
        epoch = int(layer.plan[EPOCH])
        y = layer.run_layer(x[:n], router, shared_experts=1, norm=(scale, 1e-6) if norm else None)[0]
        torch.cuda.synchronize()
        assert int(layer.plan[EPOCH]) == epoch + moved and int(layer.status[:n].sum()) == 0
        assert torch.equal(y.view(torch.int32), torch.cat(singles[:n]).view(torch.int32))


# rows whose deltas and sums (hidden / 8 bytes each) share cache lines with their neighbours' in the image that the launch writes and reads; other rows in every
# call, so that what a line held before is wrong
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(16, 256, 512, 16, 8), (16, 1280, 768, 32, 8), (13, 1792, 512, 32, 8), (16, 2304, 512, 32, 8), (11, 3328, 768, 24, 8)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rows_that_share_lines_of_the_image(strix, rows, hidden, ffn, experts, top_k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u = (blocks(gen, experts * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, experts * hidden, ffn, 256, 144, (1, 3))
    layer, staged = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    inputs = [(torch.randn((rows, hidden), device="cuda", generator=gen) * 2.0 ** (4 * i - 8)).to(dtype) for i in range(5)]
    epoch = int(layer.plan[EPOCH])
    outs = []
    for x in inputs:
        y, ids, w, _ = layer.run_layer(x, router)
        outs.append((y.clone(), ids.clone(), w.clone(), layer.status[:rows].clone()))
    assert int(layer.plan[EPOCH]) == epoch + len(inputs)
    for x, (y, ids, w, status) in zip(inputs, outs):
        want_ids, want_w = strix.route(x, router, top_k)[:2]
        assert torch.equal(ids, want_ids) and torch.equal(w.view(torch.int32), want_w.view(torch.int32)) and int(status.sum()) == 0
        assert torch.equal(y.view(torch.int32), staged.run(x, want_ids, want_w).view(torch.int32))


def wide_layer(strix, rows, hidden, ffn, experts, top_k, intermediates=False):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + ffn)
    g, u = (blocks(gen, experts * ffn, hidden, 256, 144, (1, 3)) for _ in range(2))
    d = blocks(gen, experts * hidden, ffn, 256, 144, (1, 3))
    layer, staged = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, rows, intermediates=intermediates) for _ in range(2))
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    return layer, staged, router, torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)


# experts of more than 4 MB of gate and up rows, whose assignments are swept again by helper blocks: more and fewer helpers a row than groups of 32 outputs, none, one
# and several slots of a row, an assignment that overflows on the exact expert and one that does on the early one
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(1, 2048, 2048, 16, 8), (16, 2304, 1792, 16, 8), (5, 4096, 1536, 24, 6), (3, 6144, 768, 16, 16)])
@pytest.mark.parametrize("intermediates", [False, True])
def test_repairs_by_helpers(strix, rows, hidden, ffn, experts, top_k, intermediates):
    layer, staged, router, x = wide_layer(strix, rows, hidden, ffn, experts, top_k, intermediates)
    for scale in (1.0, 2.0 ** 14):
        rows32 = x.float() * scale
        ids, w = (t.clone() for t in strix.route(rows32, router, top_k)[:2])
        layer.output.fill_(7.0)
        staged.output.fill_(7.0)
        want = staged.run(rows32, ids, w).clone()
        for displaced in (0, 20, 100, 300, 0):
            strix.lib().mi355_debug_early_route_perturb(displaced)
            try:
                y, got, _, _ = layer.run_layer(rows32, router)
                torch.cuda.synchronize()
            finally:
                strix.lib().mi355_debug_early_route_perturb(0)
            assert torch.equal(got, ids) and torch.equal(layer.status[:rows], staged.status[:rows])
            assert torch.equal(y.view(torch.int32), want.view(torch.int32)), (scale, displaced)
            assert torch.equal(layer.down_codes[:rows * top_k], staged.down_codes[:rows * top_k])


def test_a_repair_of_a_large_expert_is_shared(strix):
    """One wave sweeps 18 MB in 1.8 ms, which would be twenty times the layer."""
    layer, _, router, x = wide_layer(strix, 1, 6144, 2560, 32, 8)
    ids = strix.route(x, router, 8)[0].cpu()

    def missed(displaced):
        early = early_choice(x.float().cpu().numpy(), router.cpu().numpy(), 8, displaced)[0].tolist()
        return len(set(ids[0].tolist()) - set(early))

    def micros(displaced):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        taken = []
        strix.lib().mi355_debug_early_route_perturb(displaced)
        try:
            for _ in range(12):
                begin.record()
                layer.run_layer(x, router)
                end.record()
                torch.cuda.synchronize()
                taken.append(begin.elapsed_time(end) * 1e3)
        finally:
            strix.lib().mi355_debug_early_route_perturb(0)
        return min(taken)

    displaced = next(d for d in range(1, 400) if missed(d) == 1)
    plain, repaired = micros(0), micros(displaced)
    assert repaired < 5 * plain, (plain, repaired)
