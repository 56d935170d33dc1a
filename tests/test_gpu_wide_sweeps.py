"""The 32-row matrix-core sweeps (gate and up on one wavefront, or wide: two tiles of weight rows, eight wavefronts): chunks around the lines between their
result registers (8, 16, 24 and 32 rows), both K-quant gate formats, scales and minimums that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def blocks(strix, gen, kind, rows, width):
    if kind == "q4_k":
        return strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((rows, width), device="cuda", generator=gen) * 0.02)
    w = torch.randint(0, 256, (rows, width // 256, 176), dtype=torch.uint8, device="cuda", generator=gen)       # Q5_K: d and dmin small and finite
    for at in (1, 3):
        w[..., at] = (w[..., at] & 0x03) | 0x0C
    return w.reshape(rows, -1)


# rows of the experts (one choice a row); hidden and ffn of one super-block, of two and more, of a run of tiles; against batches of two rows,
# which other sweeps serve. The sums have one order, so the bits are the same. wide: the form of the gate / up rows by stages times rows an expert (the down
# rows are wide at hidden 3072).
@pytest.mark.parametrize("counts,hidden,ffn,wide", [
    ((1, 8, 9, 16, 17, 24, 25, 32, 33), 256, 256, False), ((128, 65, 40, 0, 41, 0), 512, 768, False), ((38, 27, 1, 14), 1792, 256, False),
    ((450, 360, 401, 395), 256, 256, True), ((200, 240, 193, 177), 512, 512, True), ((129, 31, 1, 64), 2304, 256, True), ((1, 8, 9, 16, 17, 24, 25, 32, 33), 3072, 256, True)])
@pytest.mark.parametrize("gate", ["q4_k", "q5_k"])
@pytest.mark.parametrize("special", [None, 0x7C00, 0xFC00])
def test_chunks_equal_pairs_of_rows(strix, counts, hidden, ffn, wide, gate, special):
    E, T = len(counts), sum(counts)
    stages = hidden // 256
    assert wide == (stages >= 12 or stages * T >= 400 * E if gate == "q5_k" else stages >= 8 or stages * T >= 180 * E)      # (workgroups of one tile)
    assert T >= 16 * E                                                     # the rule of items longer than 16 rows
    gen = torch.Generator(device="cuda").manual_seed(hidden + ffn)
    gt = strix.TYPE_Q4_K if gate == "q4_k" else strix.TYPE_Q5_K
    g, u, d = blocks(strix, gen, gate, E * ffn, hidden), blocks(strix, gen, gate, E * ffn, hidden), blocks(strix, gen, "q4_k", E * hidden, ffn)
    if special is not None:                                                # down rows 3 and 5 of every expert: an infinite scale, an infinite minimum
        rows = d.view(E, hidden, -1)
        for row, at in ((3, 0), (5, 2)):
            rows[:, row, at], rows[:, row, at + 1] = special & 255, special >> 8
    ids = torch.tensor([e for e, c in enumerate(counts) for _ in range(c)], dtype=torch.int32)[:, None]
    ids = ids[torch.randperm(T, generator=torch.Generator().manual_seed(1))].cuda()
    x, w = torch.randn((T, hidden), device="cuda", generator=gen).to(torch.float16), torch.rand((T, 1), device="cuda", generator=gen) + 0.5
    layer, pair = (strix.MoeLayer(hidden, ffn, E, 1, g, u, d, n, gate_type=gt) for n in (T, 2))
    out = layer.run(x, ids, w).clone()
    flag = 0 if special is None else strix.STATUS_AGGREGATE
    assert bool((layer.status[:T] == flag).all()) and (special is None) == bool(out.isfinite().all())
    for r in range(0, T - 1, 2 if T < 200 else 6):
        want = pair.run(x[r:r + 2], ids[r:r + 2].contiguous(), w[r:r + 2].contiguous())
        same = (out[r:r + 2].view(torch.int32) == want.view(torch.int32)) | (out[r:r + 2].isnan() & want.isnan())
        assert bool(same.all()), r


# a dense block: rows of one chunk and of three, few workgroups of down rows (which stay on sixteen rows a sweep) and one per compute unit
@pytest.mark.parametrize("rows,hidden,ffn", [(17, 512, 1024), (25, 256, 512), (33, 1792, 512), (48, 256, 1024), (70, 8192, 512)])
def test_dense_rows_equal_one_by_one(strix, rows, hidden, ffn):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    g, u, d = (blocks(strix, gen, "q4_k", n, m) for n, m in ((ffn, hidden), (ffn, hidden), (hidden, ffn)))
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.bfloat16)
    ids, one = torch.zeros((rows, 1), dtype=torch.int32, device="cuda"), torch.ones((rows, 1), device="cuda")
    layer, alone = (strix.MoeLayer(hidden, ffn, 1, 1, g, u, d, n, intermediates=True) for n in (rows, 1))
    out = layer.run(x, ids, one)
    for r in range(rows):
        assert torch.equal(out[r:r + 1].view(torch.int32), alone.run(x[r:r + 1], ids[:1], one[:1]).view(torch.int32)), r


# long down rows of a dense block in stage teams: both numbers of ring slots (2048 | 16384 is the least matrix of three), stages that the teams do not
# share evenly, fewer stages than teams; against batches of one row, which the vector-ALU sweeps serve
@pytest.mark.parametrize("hidden,ffn", [(256, 512), (512, 8448), (2048, 16384), (2048, 16640), (1024, 33024)])
@pytest.mark.parametrize("rows", [3, 4, 5, 8])
def test_stage_teams_equal_one_by_one(strix, hidden, ffn, rows):
    gen = torch.Generator(device="cuda").manual_seed(hidden + ffn + rows)
    draw = lambda n, m: strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    tensors = draw(ffn, hidden), draw(ffn, hidden), draw(hidden, ffn)
    layer, one = (strix.MoeLayer(hidden, ffn, 1, 1, *tensors, n, intermediates=True) for n in (rows, 1))
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(torch.float16)
    ids, weights = torch.zeros((rows, 1), dtype=torch.int32, device="cuda"), torch.ones((rows, 1), device="cuda")
    out = layer.run(x, ids, weights).clone()
    assert int(layer.status[:rows].sum()) == 0
    for r in range(rows):
        assert torch.equal(out[r:r + 1].view(torch.int32), one.run(x[r:r + 1], ids[r:r + 1], weights[r:r + 1]).view(torch.int32)), r
