"""The router of batches past the decode sizes (its chains run on the fp32 matrix cores), bit for bit against the CPU oracle."""
import numpy as np
import pytest
import torch

import orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


# rows and experts around the tiles of 16 and the workgroups of 64 experts; features around the blocks of 32 and the rings of 4 and 8
# blocks (4112 rows x 64 experts: more workgroups than compute units, the short ring)
@pytest.mark.parametrize("rows,experts,hidden,top_k", [(17, 5, 32, 2), (32, 16, 96, 4), (33, 130, 256, 8), (100, 63, 288, 6), (18, 300, 2080, 16), (64, 65, 4064, 8),
                                                       (4112, 64, 160, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_logits_of_a_batch(strix, rows, experts, hidden, top_k, dtype):
    gen = torch.Generator().manual_seed(rows + experts + hidden)
    x = torch.randn((rows, hidden), generator=gen).to(dtype)
    w = torch.randn((experts, hidden), generator=gen) * 0.05
    x[0, ::3] *= 2.0 ** -20                      # subnormal halves; products over many binades
    w[0] *= 2.0 ** -120
    bias = torch.randn(experts, generator=gen) if experts % 2 else None
    ids, weights, scores = strix.route(x.cuda(), w.cuda(), top_k, bias=None if bias is None else bias.cuda())
    ids_ref, w_ref, s_ref, _ = orc.route(x.float().numpy(), w.numpy(), top_k, bias=None if bias is None else bias.numpy())
    assert np.array_equal(bits(scores.cpu().numpy()), bits(s_ref))
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), ids_ref) and np.array_equal(bits(weights.cpu().numpy()), bits(w_ref))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_rows_of_any_values(strix, dtype):
    """Infinities, NaN, zeros of both signs and values that overflow, in the rows and in the router weights, rows with a stride: the
    bits of decode batches, whose chains run on the vector ALU."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    rows, experts, hidden, top_k = 40, 96, 1056, 4
    inf, nan = float("inf"), float("nan")
    wide = torch.randn((rows, hidden + 32), device="cuda", generator=gen)
    x = wide[:, :hidden]
    x[1, 5], x[2, 7], x[3, 9], x[4, 3], x[4, 100], x[5], x[6], x[7], x[8] = inf, -inf, nan, inf, -inf, inf, nan, 0.0, -0.0
    x[9] *= 3e38
    x[10] *= 1e-42
    x = wide.to(dtype)[:, :hidden]
    w = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    bad = w.clone()
    bad[3, 2], bad[4, 2], bad[5, 5] = inf, nan, -inf
    for router, bias in ((w, None), (w, torch.randn(experts, device="cuda", generator=gen)), (bad, None)):
        batch = strix.route(x, router, top_k, bias=bias)
        parts = [strix.route(x[r:r + 8].contiguous(), router, top_k, bias=bias) for r in range(0, rows, 8)]
        for got, want in zip(batch, zip(*parts)):
            assert torch.equal(got.view(torch.int32), torch.cat(want).view(torch.int32))


# around the lines between the rings: sixteen blocks of a workgroup of one wave (as many blocks, one less and one more; 512 and 528, 768 and 784
# waves), eight and four of a workgroup of four waves; a row's value does not depend on the batch, so decode batches state it
@pytest.mark.parametrize("rows,experts,hidden", [(40, 20, 480), (40, 20, 512), (40, 20, 544), (512, 256, 128), (513, 250, 288), (768, 256, 160), (769, 256, 544), (4097, 64, 96)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rings_of_a_batch(strix, rows, experts, hidden, dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x, w = torch.randn((rows, hidden), device="cuda", generator=gen).to(dtype), torch.randn((experts, hidden), device="cuda", generator=gen) * 0.05
    batch = strix.route(x, w, 4)
    for r in (0, rows // 2, rows - 16):
        for got, want in zip(batch, strix.route(x[r:r + 16].contiguous(), w, 4)):
            assert torch.equal(got[r:r + 16].view(torch.int32), want.view(torch.int32)), r


# decode rows past 2048 features, whose logits alone run on the matrix cores too, in two waves a tile: blocks around the meetings of the waves (every
# four blocks) and the ring's end (sixteen)
@pytest.mark.parametrize("rows,experts,hidden,top_k", [(1, 16, 2080, 2), (7, 33, 2112, 4), (16, 130, 2144, 8), (15, 20, 2176, 4), (9, 64, 2560, 8), (16, 17, 6144, 8), (3, 5, 16384, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_wide_decode_rows(strix, rows, experts, hidden, top_k, dtype):
    gen = torch.Generator().manual_seed(rows + experts + hidden)
    x = torch.randn((rows, hidden), generator=gen).to(dtype)
    w = torch.randn((experts, hidden), generator=gen) * 0.05
    x[0, ::3] *= 2.0 ** -20
    w[0] *= 2.0 ** -120
    bias = torch.randn(experts, generator=gen) if experts % 2 else None
    ids, weights, scores = strix.route(x.cuda(), w.cuda(), top_k, bias=None if bias is None else bias.cuda())
    ids_ref, w_ref, s_ref, _ = orc.route(x.float().numpy(), w.numpy(), top_k, bias=None if bias is None else bias.numpy())
    assert np.array_equal(bits(scores.cpu().numpy()), bits(s_ref))
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), ids_ref) and np.array_equal(bits(weights.cpu().numpy()), bits(w_ref))


# infinities, NaN, zeros of both signs and values that overflow in decode rows of that width: the bits of the chains that the vector ALU runs beside a layer's sweeps
@pytest.mark.parametrize("rows,hidden", [(13, 2304), (16, 4096)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_wide_decode_rows_of_any_values(strix, rows, hidden, dtype):
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden)
    experts, top_k, ffn, inf, nan = 32, 8, 256, float("inf"), float("nan")
    x = torch.randn((rows, hidden), device="cuda", generator=gen)
    x[1, 5], x[2, 2071], x[3, 9], x[4, 3], x[4, 2100], x[5], x[6], x[7], x[8] = inf, -inf, nan, inf, -inf, inf, nan, 0.0, -0.0
    x[9] *= 3e38
    x[10] *= 1e-42
    x = x.to(dtype)
    gate, up = (strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((experts * ffn, hidden), device="cuda", generator=gen)) for _ in range(2))
    down = strix.quantize_weight_rows(strix.TYPE_Q4_K, torch.randn((experts * hidden, ffn), device="cuda", generator=gen))
    layer = strix.MoeLayer(hidden, ffn, experts, top_k, gate, up, down, rows)
    w = torch.randn((experts, hidden), device="cuda", generator=gen) * 0.02
    bad = w.clone()
    bad[3, 2], bad[4, 2200], bad[5, 5] = inf, nan, -inf
    for router in (w, bad):
        scores = strix.route(x, router, top_k)[2]
        beside = layer.run_layer(x, router)[3]
        assert torch.equal(scores.reshape(-1).view(torch.int32), beside.reshape(-1)[:rows * experts].view(torch.int32))
        want = orc.route(x.float().cpu().numpy(), router.cpu().numpy(), top_k)[2]
        got = scores.cpu().numpy().reshape(want.shape)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~np.isnan(want)], want[~np.isnan(want)])
