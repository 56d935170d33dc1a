"""Workgroups of the wide fp16 prefill form over several units: lists with gaps, lists that are filled again, the last unit of each."""
import pytest
import torch

from test_gpu_prefill_formats import draw

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def tensors(strix, gen, kind, experts, hidden, ffn):
    def rows_of(rows, width):
        if kind == strix.TYPE_Q5_K:
            return draw(gen, "q5_k", rows, width)[0]
        return strix.quantize_weight_rows(kind, torch.randn((rows, width), device="cuda", generator=gen) * 0.05)
    return rows_of(experts * ffn, hidden), rows_of(experts * ffn, hidden), rows_of(experts * hidden, ffn)


# experts of no, of one to four token tiles, of a whole item and of an item and one more row
@pytest.mark.parametrize("kind", ["q4_k", "q5_k", "q8_0"])
@pytest.mark.parametrize("hidden,ffn,counts", [(512, 2304, [0, 57, 128, 129, 0, 300, 64, 200, 0, 385, 90, 257, 511]), (2048, 1280, [0, 0, 2000, 58])])
def test_units_of_uneven_experts(strix, prefill_forms, kind, hidden, ffn, counts):
    """Every row's output is what its expert alone gives it: the sums of a row do not depend on the batch nor on the form (the batch takes the wide
    one, an expert alone the four-wave form), so the bits are the same."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    kind = {"q4_k": strix.TYPE_Q4_K, "q5_k": strix.TYPE_Q5_K, "q8_0": strix.TYPE_Q8_0}[kind]
    experts, rows = len(counts), sum(counts)
    gate, up, down = tensors(strix, gen, kind, experts, hidden, ffn)
    ids = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(rows, generator=torch.Generator().manual_seed(6))].to("cuda", torch.int32).reshape(rows, 1)
    x = (torch.randn((rows, hidden), device="cuda", generator=gen) * (0.05 if kind == strix.TYPE_Q5_K else 1.0)).half()
    weights = torch.rand((rows, 1), device="cuda", generator=gen)
    layer = strix.MoeLayer(hidden, ffn, experts, 1, gate, up, down, rows, prefill_f16=True, gate_type=kind, down_type=kind)
    prefill_forms.use("wide")
    out = layer.run_prefill_f16(x, ids, weights).clone()
    prefill_forms.check(layer)
    prefill_forms.use("four_waves")
    for e, n in enumerate(counts):
        if n == 0:
            continue
        at = (ids.reshape(-1) == e).nonzero().squeeze(1)
        one = strix.MoeLayer(hidden, ffn, 1, 1, gate[e * ffn:(e + 1) * ffn], up[e * ffn:(e + 1) * ffn], down[e * hidden:(e + 1) * hidden], n,
                             prefill_f16=True, gate_type=kind, down_type=kind)
        alone = one.run_prefill_f16(x[at].contiguous(), torch.zeros((n, 1), dtype=torch.int32, device="cuda"), weights[at].contiguous())
        prefill_forms.check(one)
        assert torch.equal(out[at], alone), (e, n)
    assert int(layer.status.max()) == 0


def test_lists_are_filled_again(strix, prefill_forms):
    """More than 64 units a workgroup on 256 compute units (136 item slots of 132 tiles): bit for bit the rows in pieces."""
    gen = torch.Generator(device="cuda").manual_seed(7)
    hidden, ffn, rows, piece = 256, 16896, 16500, 5500
    gate, up, down = tensors(strix, gen, strix.TYPE_Q4_K, 1, hidden, ffn)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).half()
    ids, one = torch.zeros((rows, 1), dtype=torch.int32, device="cuda"), torch.ones((rows, 1), device="cuda")
    layer = strix.MoeLayer(hidden, ffn, 1, 1, gate, up, down, rows, prefill_f16=True)
    whole = layer.run_prefill_f16(x, ids, one)
    prefill_forms.check(layer, "wide")
    parts = strix.MoeLayer(hidden, ffn, 1, 1, gate, up, down, piece, prefill_f16=True)
    for at in range(0, rows, piece):
        assert torch.equal(whole[at:at + piece], parts.run_prefill_f16(x[at:at + piece], ids[:piece], one[:piece])), at


def test_many_experts_in_another_order(strix, prefill_form):
    """600 experts of few rows each, several items' tiles a workgroup: a batch and the same rows in another order."""
    gen = torch.Generator(device="cuda").manual_seed(8)
    hidden, ffn, rows, experts, top_k = 256, 256, 1400, 600, 8
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, *tensors(strix, gen, strix.TYPE_Q4_K, experts, hidden, ffn), rows, prefill_f16=True)
    x = torch.randn((rows, hidden), device="cuda", generator=gen).half()
    ids = (torch.rand((rows, experts), device="cuda", generator=gen) + torch.linspace(0, 1, experts, device="cuda")).topk(top_k).indices.int()
    weights = torch.rand((rows, top_k), device="cuda", generator=gen)
    out = layer.run_prefill_f16(x, ids, weights).clone()
    prefill_form.check(layer)
    assert torch.equal(layer.run_prefill_f16(x.flip(0), ids.flip(0), weights.flip(0)).flip(0), out)


@pytest.mark.parametrize("kind", ["q4_k", "q5_k"])
def test_workspace_of_nan(strix, prefill_form, kind):
    """Sums past a row's sub-blocks (hidden 1280 and ffn 768 leave eight slots of a group of sixteen) and rows of h past an item's are read and never part of a
    value: a workspace full of NaN gives the bits of a clean one."""
    gen = torch.Generator(device="cuda").manual_seed(9)
    hidden, ffn, rows, experts, top_k = 1280, 768, 150, 4, 2
    kind = {"q4_k": strix.TYPE_Q4_K, "q5_k": strix.TYPE_Q5_K}[kind]
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, *tensors(strix, gen, kind, experts, hidden, ffn), rows, prefill_f16=True, gate_type=kind, down_type=kind)
    x = (torch.randn((rows, hidden), device="cuda", generator=gen) * 0.05).half()
    ids = torch.rand((rows, experts), device="cuda", generator=gen).topk(top_k).indices.int()
    weights = torch.rand((rows, top_k), device="cuda", generator=gen)
    layer.h_f16.zero_()
    want = layer.run_prefill_f16(x, ids, weights).clone()
    layer.h_f16.fill_(0xFF)
    assert torch.equal(layer.run_prefill_f16(x, ids, weights), want) and int(layer.status[:rows].sum()) == 0
    prefill_form.check(layer)
