"""The start of a staged batch: the plan's order around the limit of its one workgroup, and the launch that selects, checks and quantises a row."""
import numpy as np
import pytest
import torch

import orc

pytestmark = pytest.mark.gpu

PLAN_OFFSETS_AT = 2240          # first word of the plan arrays (offsets, touched, order, items)


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def pad4(n):
    return (n + 3) // 4 * 4


# assignments around a wave's 64, around 1024 (an assignment per thread of the plan's one workgroup) and past it (a workgroup per expert); one expert that
# takes everything (skew 2), more experts than assignments, ids of no expert (skew 3)
@pytest.mark.parametrize("rows,top_k,experts,skew", [(1, 1, 2, 0), (1, 1, 1, 0), (63, 1, 5, 0), (64, 1, 1024, 0), (65, 1, 3, 2), (32, 8, 128, 0), (257, 1, 16, 1), (341, 3, 40, 0),
                                                     (64, 16, 300, 2), (64, 16, 1024, 0), (1025, 1, 64, 1), (205, 5, 7, 0), (2049, 1, 1, 0), (100, 16, 1024, 0),
                                                     (40, 8, 31, 3), (128, 8, 1023, 3), (200, 8, 64, 3)])
def test_plan_order(strix, rows, top_k, experts, skew):
    rng = np.random.default_rng(rows * top_k + experts)
    ids = np.minimum(rng.integers(0, experts, (rows, top_k)), rng.integers(0, experts, (rows, top_k)) // (1 if skew == 0 else 4)) if skew < 2 else np.full((rows, top_k), experts - 1)
    if skew == 3:
        ids = rng.integers(0, experts, (rows, top_k))
        ids.reshape(-1)[::7] = experts + rng.integers(0, 2000, ids.reshape(-1)[::7].shape)
    H = I = 256
    row = H // 256 * 144
    w = torch.zeros((experts * 256, row), dtype=torch.uint8, device="cuda")
    layer = strix.MoeLayer(H, I, experts, top_k, w, w, w, rows)
    x = torch.zeros((rows, H), device="cuda")
    routes = torch.from_numpy(ids.astype(np.int32)).cuda()
    layer.stage("csr", x, routes, torch.ones((rows, top_k), device="cuda"))
    plan = layer.plan.cpu().numpy()
    flat, A = ids.reshape(-1), rows * top_k
    live = np.flatnonzero(flat < experts)
    order_at = PLAN_OFFSETS_AT + pad4(experts + 1) + pad4(experts)
    offsets = np.concatenate([[0], np.cumsum(np.bincount(flat[live], minlength=experts))])
    assert np.array_equal(plan[PLAN_OFFSETS_AT:PLAN_OFFSETS_AT + experts + 1], offsets)
    assert plan[0] == A and plan[1] == len(set(flat[live])) and plan[2] == np.diff(offsets).max()
    assert np.array_equal(plan[PLAN_OFFSETS_AT + pad4(experts + 1):][:plan[1]], np.unique(flat[live]))
    assert np.array_equal(plan[order_at:order_at + len(live)], live[np.argsort(flat[live], kind="stable")])
    items = plan[order_at + pad4(A):][:4 * plan[4]].reshape(-1, 4)
    covered = np.concatenate([np.arange(b, e) for _, b, e, _ in items])
    assert np.array_equal(covered, np.arange(len(live))) and all(offsets[e] <= b < z <= offsets[e + 1] for e, b, z, _ in items)


# the plan that is made beside the rows of a batch, in the launch that quantises them or sums them for the prefill: around a turn of 64 assignments a
# wavefront, the eight turns it asks for together and more; experts that nothing chose, ids of no expert
@pytest.mark.parametrize("rows,top_k,experts", [(3, 1, 2), (17, 4, 1024), (65, 4, 5), (513, 8, 300), (600, 16, 40), (4200, 3, 3)])
@pytest.mark.parametrize("prefill", [False, True])
def test_plan_beside_the_rows(strix, rows, top_k, experts, prefill):
    rng = np.random.default_rng(rows + experts)
    ids = np.minimum(rng.integers(0, experts, (rows, top_k)), rng.integers(0, experts, (rows, top_k)))
    ids[rows // 2, 0] = experts + 3
    H = I = 256
    w = torch.zeros((experts * 256, 144), dtype=torch.uint8, device="cuda")
    layer = strix.MoeLayer(H, I, experts, top_k, w, w, w, rows, prefill_f16=prefill)
    x, routes, ones = torch.zeros((rows, H), device="cuda", dtype=torch.float16), torch.from_numpy(ids.astype(np.int32)).cuda(), torch.ones((rows, top_k), device="cuda")
    (layer.run_prefill_f16 if prefill else layer.run)(x, routes, ones)
    plan = layer.plan.cpu().numpy()
    flat, A = ids.reshape(-1), rows * top_k
    counts = np.bincount(flat[flat < experts], minlength=experts)
    offsets, order_at = np.concatenate([[0], np.cumsum(counts)]), PLAN_OFFSETS_AT + pad4(experts + 1) + pad4(experts)
    assert plan[0] == A and plan[1] == np.count_nonzero(counts) and plan[2] == counts.max()
    assert np.array_equal(plan[PLAN_OFFSETS_AT:PLAN_OFFSETS_AT + experts + 1], offsets)
    assert np.array_equal(plan[PLAN_OFFSETS_AT + pad4(experts + 1):][:plan[1]], np.nonzero(counts)[0])
    order = np.argsort(np.where(flat < experts, flat, experts), kind="stable")[:A - 1]
    assert np.array_equal(plan[order_at:order_at + A - 1], order)
    items = plan[order_at + pad4(A):][:4 * plan[4]].reshape(-1, 4)
    assert np.array_equal(np.concatenate([np.arange(b, e) for _, b, e, _ in items]), np.arange(A - 1)) and all(offsets[e] <= b < z <= offsets[e + 1] for e, b, z, _ in items)
    assert [bool(s & strix.STATUS_INVALID_ROUTE) for s in layer.status[:rows].cpu().tolist()] == [r == rows // 2 for r in range(rows)]


# widths around the image's 448 threads of eight values; experts around the selection's register steps; a row with an infinity
# (its weights are not finite either: both status bits), rows past and within the decode sizes (large experts: shared sweeps)
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(17, 256, 256, 5, 2), (40, 3584, 256, 130, 8), (33, 3840, 256, 16, 4), (18, 8192, 256, 20, 16), (16, 6144, 1280, 24, 8)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_layer_equals_router_then_experts(strix, rows, hidden, ffn, experts, top_k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    draw = lambda n, m: strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, draw(experts * ffn, hidden), draw(experts * ffn, hidden), draw(experts * hidden, ffn), rows)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(dtype)
    x[rows // 2, hidden - 1] = float("inf")
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    out, ids, weights, scores = (t.clone() for t in layer.run_layer(x, router))
    status = layer.status[:rows].clone()
    ids2, weights2, scores2 = strix.route(x, router, top_k)
    same = lambda a, b: torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))
    assert same(ids, ids2) and same(weights, weights2) and same(scores, scores2)
    out2 = layer.run(x, ids2, weights2)
    good = torch.arange(rows, device="cuda") != rows // 2
    assert same(out[good], out2[good]) and same(status, layer.status[:rows])
    bad = strix.STATUS_NONFINITE_ACTIVATION | strix.STATUS_INVALID_ROUTE
    assert [s & bad for s in status.cpu().tolist()] == [bad if r == rows // 2 else 0 for r in range(rows)]
    ids_ref, w_ref, _, _ = orc.route(x[:1].float().cpu().numpy(), router.cpu().numpy(), top_k)
    assert np.array_equal(ids[:1].cpu().numpy().astype(np.uint32), ids_ref) and np.array_equal(weights[:1].cpu().numpy().view(np.uint32), w_ref.view(np.uint32))
    layer.run(x, torch.full_like(ids2, experts), weights2 * 0 + 1)          # routes outside the experts
    assert all(s & strix.STATUS_INVALID_ROUTE for s in layer.status[:rows].cpu().tolist())


# the four-wave prefill with experts of one row, around 32, 64 and 128 rows, against the wide form on each expert alone
@pytest.mark.parametrize("counts,hidden,ffn", [((1, 64, 0, 65, 31, 0, 32, 0, 0, 0, 0, 0), 256, 768), ((128, 0, 0, 0, 33, 1, 0, 0, 0, 0, 0, 0), 512, 256),
                                               ((129, 63, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0), 1280, 768)])
def test_narrow_prefill_equals_wide(strix, prefill_forms, counts, hidden, ffn):
    E = len(counts)
    gen = torch.Generator(device="cuda").manual_seed(hidden)
    draw = lambda n, m: strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    gate, up, down = draw(E * ffn, hidden), draw(E * ffn, hidden), draw(E * hidden, ffn)
    ids = torch.tensor([e for e, c in enumerate(counts) for _ in range(c)], dtype=torch.int32)[:, None]
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(1))].cuda()
    T = len(ids)
    x = torch.randn((T, hidden), device="cuda", generator=gen).to(torch.float16)
    ones = torch.ones((T, 1), device="cuda")
    prefill_forms.use("four_waves")
    layer = strix.MoeLayer(hidden, ffn, E, 1, gate, up, down, T, prefill_f16=True)
    narrow = layer.run_prefill_f16(x, ids, ones)
    prefill_forms.check(layer)
    prefill_forms.use("wide")
    for e in {int(i) for i in ids.flatten()}:                              # expert by expert as one-expert layers
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        pick = lambda t, n: t[e * n:(e + 1) * n].contiguous()
        alone = strix.MoeLayer(hidden, ffn, 1, 1, pick(gate, ffn), pick(up, ffn), pick(down, hidden), len(rows), prefill_f16=True)
        got = alone.run_prefill_f16(x[rows].contiguous(), torch.zeros_like(ids[rows]), ones[rows])
        prefill_forms.check(alone)
        assert torch.equal(got, narrow[rows])                              # the same products and sums in the same order


# rows per expert around the lines between items of 4, 8, 16 and 128 rows (3, 12 and 16 rows per expert; 8 with another down format), experts
# with none and with all of the rows, decode batches over large experts (3 and 16 rows more than the small-batch sweeps take); against
# batches of two rows, which the vector-ALU sweeps serve
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k,down", [(17, 512, 256, 40, 2, "q4_k"), (23, 256, 512, 16, 2, "q4_k"), (24, 512, 256, 16, 2, "q4_k"), (95, 256, 256, 8, 1, "q4_k"),
                                                                (96, 512, 256, 8, 1, "q4_k"), (65, 256, 256, 8, 2, "q4_k"), (31, 512, 256, 8, 2, "q6_k"), (33, 256, 512, 8, 2, "q8_0"),
                                                                (33, 256, 256, 40, 8, "q5_1"), (13, 4096, 1024, 12, 4, "q4_k"), (16, 3072, 1280, 30, 8, "q4_k")])
@pytest.mark.parametrize("skew", [False, True])
def test_batches_equal_pairs_of_rows(strix, rows, hidden, ffn, experts, top_k, down, skew):
    gen = torch.Generator(device="cuda").manual_seed(rows * hidden + skew)
    kind = {"q4_k": strix.TYPE_Q4_K, "q6_k": strix.TYPE_Q6_K, "q8_0": strix.TYPE_Q8_0, "q5_1": strix.TYPE_Q5_1}[down]
    draw = lambda t, n, m: strix.quantize_weight_rows(t, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    if down in ("q4_k", "q8_0"):
        wd = draw(kind, experts * hidden, ffn)
    else:                                                                  # random blocks with small finite scales
        size, per, scales, high = {"q6_k": (210, 256, (209,), 0x08), "q5_1": (24, 32, (1, 3), 0x14)}[down]
        wd = torch.randint(0, 256, (experts * hidden, ffn // per, size), dtype=torch.uint8, device="cuda", generator=gen)
        for at in scales:
            wd[..., at] = (wd[..., at] & 0x03) | high
        wd = wd.reshape(experts * hidden, -1)
    gate, up = draw(strix.TYPE_Q4_K, experts * ffn, hidden), draw(strix.TYPE_Q4_K, experts * ffn, hidden)
    gate.view(-1, 144)[5, :2] = torch.tensor([0x00, 0x7C], dtype=torch.uint8, device="cuda")           # one infinite scale: a flagged projection
    make = lambda n: strix.MoeLayer(hidden, ffn, experts, top_k, gate, up, wd, n, down_type=kind)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)
    score = torch.rand((rows, experts), device="cuda", generator=gen)
    if skew:
        score[:, experts - top_k:] += 2.0                                  # every row on the same experts, none of them expert 0
    score[:, 0] = -1.0                                                     # (expert 0 holds the infinite scale)
    ids = score.topk(top_k, dim=1).indices.to(torch.int32)
    w = torch.rand((rows, top_k), device="cuda", generator=gen)
    layer, pair = make(rows), make(2)
    same = lambda a, b: torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))
    out = layer.run(x, ids, w)
    assert int(layer.status[:rows].sum()) == 0
    for r in range(0, rows - 1, max(2, rows // 8)):
        assert same(out[r:r + 2], pair.run(x[r:r + 2], ids[r:r + 2].contiguous(), w[r:r + 2].contiguous()))
    ids[rows // 2, 0] = 0
    layer.run(x, ids, w)
    nonfinite = strix.STATUS_NONFINITE_PROJECTION
    assert [s & nonfinite for s in layer.status[:rows].cpu().tolist()] == [nonfinite if r == rows // 2 else 0 for r in range(rows)]


def test_batches_inside_a_captured_graph(strix):
    """A staged layer with its router, a narrow prefill and a projection of many rows in one graph: every replay gives the eager bits,
    with eager calls in between."""
    gen = torch.Generator(device="cuda").manual_seed(11)
    hidden, ffn, experts, top_k, rows = 512, 256, 16, 4, 40
    draw = lambda n, m: strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    tensors = draw(experts * ffn, hidden), draw(experts * ffn, hidden), draw(experts * hidden, ffn)
    layer, prompt = strix.MoeLayer(hidden, ffn, experts, top_k, *tensors, rows), strix.MoeLayer(hidden, ffn, experts, top_k, *tensors, rows, prefill_f16=True)
    router = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    w8 = strix.quantize_weight_rows(strix.TYPE_Q8_0, torch.randn((96, hidden), device="cuda", generator=gen))
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)

    def program():
        y, ids, weights, scores = layer.run_layer(x, router)
        codes, deltas, sums, status = strix.quantize_a8(x)
        return [y, ids, weights, scores, prompt.run_prefill_f16(x, ids, weights), strix.gemv_q8_0_a8(w8, codes, deltas, hidden, 96), codes, deltas, sums, status]

    want = [t.clone() for t in program()]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        program()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = program()
    for turn in range(4):
        for t in got:
            t.fill_(1)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), turn
        layer.run_layer(x[: rows - turn].contiguous(), router)
        torch.cuda.synchronize()
