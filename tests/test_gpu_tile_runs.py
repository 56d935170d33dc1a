"""Runs of weight tiles on the matrix-core sweeps: a workgroup that goes on to the next tiles gives the values of one that starts anew."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


# runs of gate / up tiles (rows of one super-block, the last run shorter) and of down tiles (one super-block, two, three: the ring's three
# slots), items of four rows, of sixteen and longer than one sweep; against batches of two rows, which the vector-ALU sweeps serve
@pytest.mark.parametrize("rows,hidden,ffn,experts,top_k", [(34, 256, 2560, 64, 4), (34, 4352, 256, 64, 4), (40, 2304, 512, 64, 8), (34, 4608, 768, 64, 4), (100, 16384, 256, 32, 2),
                                                           (300, 16384, 256, 16, 2), (300, 256, 4864, 16, 2)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_runs_equal_pairs_of_rows(strix, rows, hidden, ffn, experts, top_k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + ffn)
    draw = lambda n, m: strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((n, m), device="cuda", generator=gen) * 0.02)
    gate, up, down = draw(experts * ffn, hidden), draw(experts * ffn, hidden), draw(experts * hidden, ffn)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).to(dtype)
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k, dim=1).indices.to(torch.int32)
    w = torch.rand((rows, top_k), device="cuda", generator=gen)
    layer, pair = (strix.MoeLayer(hidden, ffn, experts, top_k, gate, up, down, n) for n in (rows, 2))
    out = layer.run(x, ids, w)
    assert int(layer.status[:rows].sum()) == 0
    for r in range(0, rows - 1, max(2, rows // 8)):
        want = pair.run(x[r:r + 2], ids[r:r + 2].contiguous(), w[r:r + 2].contiguous())
        assert torch.equal(out[r:r + 2].view(torch.int32), want.view(torch.int32)), r
