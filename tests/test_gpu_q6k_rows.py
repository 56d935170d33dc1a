"""Q6_K down rows by direct loads (down + combine in one launch, and rows that are not back to back): the oracle's bits."""
import numpy as np
import pytest
import torch

import orc
from test_gpu_parity import bits, dev, make_layer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


# blocks: super-blocks a row, around the three that are asked for together. Weights, scales and factors at the ends of their ranges: group integers of up to
# 2 * 16 * 32 * 128 * 127 (their fourfold is what is converted), factors that are subnormal in fp16. pad: bytes between rows, 2-byte aligned either way.
@pytest.mark.parametrize("blocks,rows,top_k,pad", [(1, 1, 8, 0), (2, 3, 4, 2), (3, 2, 8, 0), (4, 5, 3, 6), (5, 1, 9, 2), (7, 2, 8, 10)])
@pytest.mark.parametrize("entry", ["layer", "staged"])
def test_extreme_blocks(strix, blocks, rows, top_k, pad, entry):
    H, I, E = 256, 256 * blocks, 12
    rng = np.random.default_rng(10 * blocks + rows)
    gate, up, _ = make_layer(rng, H, I, E)
    down = orc.random_q6_k(rng, (E, H), I).reshape(E, H, blocks, 210)
    kind = rng.integers(0, 4, (E, H, blocks))
    down[kind == 0, :192] = 0                                               # every weight -32
    down[kind == 1, :192] = 255                                             # every weight 31
    down[kind < 2, 192:208] = rng.choice(np.array([127, 128], np.uint8), (int((kind < 2).sum()), 16))
    down[kind == 2, 208:210] = np.array([3, 0], np.uint8)                   # 3 * 2^-24
    down = np.ascontiguousarray(down.reshape(E, H, blocks * 210))
    row = blocks * 210 + pad
    stored = np.zeros((E, H, row), np.uint8)
    stored[:, :, :blocks * 210] = down
    x = rng.standard_normal((rows, H)).astype(np.float16)
    wr = (rng.standard_normal((E, H)) * 0.02).astype(np.float32)
    ids, weights, _, _ = orc.route(x.astype(np.float32), wr, top_k)
    layer = strix.MoeLayer(H, I, E, top_k, dev(gate), dev(up), dev(stored), rows, intermediates=True, down_type=orc.Q6_K, gate_expert_stride=I * (H // 256) * 144,
                           gate_row_stride=(H // 256) * 144, down_expert_stride=H * row, down_row_stride=row)
    y = layer.run_layer(dev(x), dev(wr))[0] if entry == "layer" else layer.run(dev(x), dev(ids.astype(np.int32)), dev(weights))
    n = rows * top_k
    image = tuple(t[:n].cpu().numpy() for t in (layer.down_codes, layer.down_deltas, layer.down_sums))
    codes, deltas, sums, _ = orc.quantize_a8(x.astype(np.float32))
    want = orc.routed_experts(H, I, top_k, gate, up, down, orc.Q6_K, codes, deltas, sums, ids, down_only_from=image)
    raw = layer.rawdots[:rows].cpu().numpy()
    assert np.array_equal(bits(raw), bits(want.rawdots))
    assert np.array_equal(bits(y.cpu().numpy()), bits(orc.combine(0, weights, ids, raw)))
