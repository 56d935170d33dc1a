"""Q5_K gate / up rows and Q6_K, Q8_0, Q5_1 down rows on the matrix-core sweeps: the values of the sweeps that serve few rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def blocks(gen, kind, rows, width):
    """Random blocks; every code and scale value occurs, the fp16 factors are small and finite."""
    per, size, scales = {"q4_k": (256, 144, (1, 3)), "q5_k": (256, 176, (1, 3)), "q6_k": (256, 210, (209,)), "q8_0": (32, 34, (1,)), "q5_1": (32, 24, (1, 3))}[kind]
    w = torch.randint(0, 256, (rows, width // per, size), dtype=torch.uint8, device="cuda", generator=gen)
    for at in scales:
        w[..., at] = (w[..., at] & 0x03) | 0x0C
    return w.reshape(rows, -1)


# items of four rows, of sixteen in sweeps of eight and of sixteen, longer than a sweep; down rows of one stage, of fewer and of more than the
# ring's slots, once enough of them that a Q6_K block starts at every even place of sixteen bytes; a decode batch over
# experts of several MB
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(17, 256, 256, 64, 4), (40, 512, 768, 16, 3), (60, 256, 1024, 16, 4), (150, 1024, 512, 8, 2), (33, 256, 2560, 32, 2),
                                                           (14, 4096, 1024, 8, 4)])
@pytest.mark.parametrize("gate,down", [("q4_k", "q6_k"), ("q4_k", "q8_0"), ("q5_k", "q5_1"), ("q5_k", "q4_k"), ("q5_k", "q8_0")])
def test_batch_equals_pairs_of_rows(strix, rows, hidden, ffn, experts, top_k, gate, down):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + ffn)
    g, u, d = blocks(gen, gate, experts * ffn, hidden), blocks(gen, gate, experts * ffn, hidden), blocks(gen, down, experts * hidden, ffn)
    x = torch.randn((rows, hidden), device="cuda", generator=gen)
    x[3] = 0.0
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k, dim=1).indices.to(torch.int32)
    w = torch.rand((rows, top_k), device="cuda", generator=gen)
    kinds = dict(gate_type=getattr(strix, "TYPE_" + gate.upper()), down_type=getattr(strix, "TYPE_" + down.upper()))
    layer, pair = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, n, **kinds) for n in (rows, 2))
    out = layer.run(x, ids, w)
    assert int(layer.status[:rows].sum()) == 0
    for r in range(0, rows - 1, max(1, rows // 12)):
        want = pair.run(x[r:r + 2], ids[r:r + 2].contiguous(), w[r:r + 2].contiguous())
        assert torch.equal(out[r:r + 2].view(torch.int32), want.view(torch.int32)), r


@pytest.mark.parametrize("gate", ["q4_k", "q5_k"])
def test_half_a_stage(strix, gate):
    """ffn 384: Q5_1 down rows keep their own sweep, the gate / up rows run here."""
    test_batch_equals_pairs_of_rows(strix, 80, 256, 384, 8, 2, gate, "q5_1")


# a dense bundle may hold its factors and code sums at any word, which the sweeps' copies do not take: the same values from the sweeps that
# read them word by word, over the batch's own plan (items of four, sixteen and more rows, and those of a layer with an always-on expert)
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(17, 256, 256, 64, 4), (60, 256, 512, 16, 4), (150, 512, 512, 8, 2), (14, 4096, 1024, 8, 4)])
@pytest.mark.parametrize("gate,down", [("q4_k", "q4_k"), ("q4_k", "q6_k"), ("q5_k", "q8_0"), ("q5_k", "q5_1")])
def test_factors_at_any_word(strix, rows, hidden, ffn, experts, top_k, gate, down):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    g, u, d = blocks(gen, gate, experts * ffn, hidden), blocks(gen, gate, experts * ffn, hidden), blocks(gen, down, experts * hidden, ffn)
    kinds = dict(gate_type=getattr(strix, "TYPE_" + gate.upper()), down_type=getattr(strix, "TYPE_" + down.upper()))

    def pair(n):
        layer, moved = (strix.MoeLayer(hidden, ffn, experts, top_k, g, u, d, n, **kinds) for _ in range(2))
        for name in ("deltas", "sums", "down_deltas", "down_sums"):
            own = getattr(moved, name)
            setattr(moved, name, torch.zeros(own.numel() + 1, dtype=own.dtype, device="cuda")[1:].reshape(own.shape))
            assert getattr(moved, name).data_ptr() % 16 == 4
        return layer, moved

    x = torch.randn((rows, hidden), device="cuda", generator=gen)
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k, dim=1).indices.to(torch.int32)
    w = torch.rand((rows, top_k), device="cuda", generator=gen)
    layer, moved = pair(rows)
    want = layer.run(x, ids, w)
    assert torch.equal(moved.run(x, ids, w).view(torch.int32), want.view(torch.int32))
    assert int(layer.status.sum()) == 0 and int(moved.status.sum()) == 0
    router = torch.randn((experts - 1, hidden), device="cuda", generator=gen) * 0.02
    layer, moved = pair(5)
    want = layer.run_layer(x[:5], router, shared_experts=1)[0]
    assert torch.equal(moved.run_layer(x[:5], router, shared_experts=1)[0].view(torch.int32), want.view(torch.int32))
