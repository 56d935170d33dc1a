"""The Q8_0 linear operators over their ranges: the A8 image of rows of every width and the product of many rows on the matrix cores,
bit for bit against the CPU oracle."""
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


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("rows,width", [(1, 32), (3, 96), (2, 2048), (5, 8192), (2, 8224), (70, 1056)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_a8_image_of_rows(strix, rows, width, dtype):
    gen = torch.Generator().manual_seed(rows * width)
    x = torch.randn((rows, width), generator=gen)
    x[0, :32] = 0.0
    x[-1, -32:] *= 2.0 ** -125
    x = x.to(dtype)
    x[rows // 2, width // 2] = float("inf")
    padded = torch.zeros((rows, width + 3), dtype=dtype)       # rows that are not 16-byte aligned: the unvectorised form
    padded[:, 1:1 + width] = x
    want = [orc.quantize_a8(r[None]) for r in x.float().numpy()]
    for view in (x.cuda(), padded.cuda()[:, 1:1 + width]):
        codes, deltas, sums, status = strix.quantize_a8(view)
        assert status.cpu().tolist() == [strix.STATUS_NONFINITE_ACTIVATION if r == rows // 2 else 0 for r in range(rows)]
        for r, (c, d, s, _) in enumerate(want):
            if r == rows // 2:
                continue
            assert np.array_equal(codes[r].cpu().numpy(), c[0]) and np.array_equal(bits(deltas[r].cpu().numpy()), bits(d[0]))
            assert np.array_equal(sums[r].cpu().numpy(), s[0])


# rows around the matrix-core form's tiles of 32 and 64, outputs around its tiles of 32 and 64, groups around its chunks of 32 (odd
# numbers of chunks, a last chunk of one group), one width whose rows are only 2-byte aligned
@pytest.mark.parametrize("rows,width,count", [(16, 1024, 70), (17, 32, 1), (32, 1056, 33), (33, 2432, 31), (64, 1024, 65), (65, 2048, 96), (130, 992, 129),
                                              (500, 64, 513), (257, 4096, 320), (40, 8192, 40), (1000, 1088, 1100)])
def test_products_of_many_rows(strix, rows, width, count):
    rng = np.random.default_rng(rows + width)
    w = orc.quantize_rows(orc.Q8_0, (rng.standard_normal((count, width)) * 0.02).astype(np.float32))
    codes, deltas, _, _ = orc.quantize_a8(rng.standard_normal((rows, width)).astype(np.float32))
    want, _ = orc.gemv_q8_0_a8(w, codes, deltas, width, count, threads=8)
    got = strix.gemv_q8_0_a8(dev(w), dev(codes), dev(deltas), width, count).cpu().numpy()
    assert np.array_equal(bits(got), bits(want))
    shifted = torch.zeros(w.size + 2, dtype=torch.uint8, device="cuda")      # weights at a pointer that is only 2-byte aligned
    shifted[2:] = dev(w).reshape(-1)
    out = torch.full((rows, count + 5), 3.0, device="cuda")
    strix.gemv_q8_0_a8(shifted[2:], dev(codes), dev(deltas), width, count, out=out, accumulate=True)
    got = out.cpu().numpy()
    assert np.array_equal(bits(got[:, :count]), bits(want + np.float32(3.0))) and np.all(got[:, count:] == 3.0)


def test_products_of_full_range_codes_and_wide_factors(strix):
    """Weight bytes of the whole int8 range and scales over many binades: the largest dots (32 * 128 * 127) and subnormal factors."""
    rng = np.random.default_rng(3)
    rows, width, count = 70, 1536, 96
    w = rng.integers(0, 256, (count, width // 32, 34), dtype=np.uint8)
    w[..., 1] = rng.integers(0, 0x78, w[..., 1].shape)         # finite scales, subnormal ones among them
    w[:4, :, 2:] = 0x80
    codes = rng.integers(-127, 128, (rows, width)).astype(np.int8)
    codes[:3] = -127
    deltas = np.exp2(rng.uniform(-120, 10, (rows, width // 32))).astype(np.float32)
    want, _ = orc.gemv_q8_0_a8(w.reshape(count, -1), codes, deltas, width, count, threads=8)
    got = strix.gemv_q8_0_a8(dev(w.reshape(count, -1)), dev(codes), dev(deltas), width, count).cpu().numpy()
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("rows", [1, 9, 40, 300])
def test_products_of_width_zero(strix, rows):
    """An empty reduction is +0 stored, or the accumulated value left as it is, for any number of rows."""
    count = 70
    w, codes = torch.zeros((count, 34), dtype=torch.uint8, device="cuda"), torch.ones((rows, 32), dtype=torch.int8, device="cuda")
    deltas = torch.ones((rows, 1), device="cuda")
    out = torch.full((rows, count), 3.0, device="cuda")
    strix.gemv_q8_0_a8(w, codes, deltas, 0, count, out=out, row_bytes_=34, accumulate=True)
    assert torch.all(out == 3.0)
    strix.gemv_q8_0_a8(w, codes, deltas, 0, count, out=out, row_bytes_=34)
    assert np.all(bits(out.cpu().numpy()) == 0)


def test_products_of_any_factors(strix):
    """Infinite, NaN, zero and negative factors, activation rows with a stride, weight rows with padding: the row sweep's values (which
    NaN survives where two meet is open)."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    rows, width, count = 40, 1056, 100
    blocks = strix.quantize_weight_rows(strix.TYPE_Q8_0, torch.randn((count, width), device="cuda", generator=gen) * 0.02).reshape(count, -1, 34)
    for o, half in enumerate((0x7C00, 0xFC00, 0x7E00, 0x0000, 0x8000), start=1):
        blocks[o, o, 0], blocks[o, o, 1] = half & 255, half >> 8
    w = torch.zeros((count, width // 32 * 34 + 6), dtype=torch.uint8, device="cuda")
    w[:, :-6] = blocks.reshape(count, -1)
    codes = torch.randint(-127, 128, (rows, width + 64), dtype=torch.int8, device="cuda", generator=gen)
    deltas = torch.rand((rows, (width + 64) // 32), device="cuda", generator=gen)
    deltas[1, 3], deltas[2, 5], deltas[3, 6], deltas[4, 7], deltas[5], deltas[6], deltas[7] = float("inf"), float("nan"), -float("inf"), 0.0, 3e38, -1.0, -0.0
    codes[8, :32], deltas[8, 0] = 0, float("inf")
    product = lambda r0, r1: strix.gemv_q8_0_a8(w, codes[r0:r1], deltas[r0:r1], width, count, row_bytes_=w.shape[1])
    want = torch.cat([product(r, r + 8) for r in range(0, rows, 8)])
    for n in (9, 32, 33, 40):
        got = product(0, n)
        assert torch.equal(got.isnan(), want[:n].isnan())
        clean = ~got.isnan()
        assert torch.equal(got[clean].view(torch.int32), want[:n][clean].view(torch.int32))


# around the lines between one, two, four and eight rows to a workgroup of the row sweep and the tiles: 768 workgroups of one and of two rows, 1536 and 1280 of
# four, 2^25 weights (five to eight rows: one round of tiles three quarters full, full and partial rounds), 256 tiles of 32 x 32 and of 32 x 64; tiles with remainders of rows, outputs and groups, of full-range codes and factors over many binades
@pytest.mark.parametrize("rows,width,count", [(3, 64, 2048), (3, 64, 2056), (8, 1056, 768), (8, 96, 776), (6, 64, 2049), (8, 64, 6144), (8, 64, 6145), (16, 1056, 769),
                                              (9, 1056, 3408), (9, 1056, 3416), (17, 32, 2177), (32, 992, 1301), (33, 2432, 1163), (70, 1536, 700), (257, 1056, 193),
                                              (5, 4096, 8191), (5, 4128, 8193), (7, 4096, 7168), (500, 2080, 1111), (33, 992, 4096), (33, 992, 4129), (100, 96, 2081),
                                              (300, 1056, 833), (200, 96, 2050), (5, 1024, 28673), (8, 2048, 14337), (6, 2048, 16383), (8, 4096, 12321), (7, 8192, 4095), (8, 6144, 6113),
                                              (5, 6144, 6145), (427, 992, 2195), (800, 96, 1280)])
def test_lines_of_the_products(strix, rows, width, count):
    rng = np.random.default_rng(rows + count)
    w = rng.integers(0, 256, (count, width // 32, 34), dtype=np.uint8)
    w[..., 1] = rng.integers(0, 0x78, w[..., 1].shape)
    codes = rng.integers(-127, 128, (rows, width)).astype(np.int8)
    deltas = np.exp2(rng.uniform(-120, 10, (rows, width // 32))).astype(np.float32)
    want, _ = orc.gemv_q8_0_a8(w.reshape(count, -1), codes, deltas, width, count, threads=8)
    shifted = torch.zeros(w.size + 2, dtype=torch.uint8, device="cuda")
    shifted[2:] = dev(w).reshape(-1)
    for weights in (dev(w.reshape(count, -1)), shifted[2:]):
        got = strix.gemv_q8_0_a8(weights, dev(codes), dev(deltas), width, count).cpu().numpy()
        assert np.array_equal(bits(got), bits(want))


def test_tiles_of_any_factors(strix):
    """Infinite, NaN, zero and negative factors on the tiles against the row sweep (which NaN survives where two meet is open)."""
    gen = torch.Generator(device="cuda").manual_seed(6)
    rows, width, count = 300, 1056, 1100
    w = strix.quantize_weight_rows(strix.TYPE_Q8_0, torch.randn((count, width), device="cuda", generator=gen) * 0.02).reshape(count, -1, 34)
    for o, half in enumerate((0x7C00, 0xFC00, 0x7E00, 0x0000, 0x8000), start=1):
        w[o, o, 0], w[o, o, 1] = half & 255, half >> 8
    codes = torch.randint(-127, 128, (rows, width), dtype=torch.int8, device="cuda", generator=gen)
    deltas = torch.rand((rows, width // 32), device="cuda", generator=gen)
    deltas[1, 3], deltas[2, 5], deltas[3, 6], deltas[4, 7], deltas[5], deltas[6], deltas[7] = float("inf"), float("nan"), -float("inf"), 0.0, 3e38, -1.0, -0.0
    codes[8, :32], deltas[8, 0] = 0, float("inf")
    product = lambda r0, r1: strix.gemv_q8_0_a8(w.reshape(count, -1), codes[r0:r1], deltas[r0:r1], width, count)
    want = torch.cat([product(r, min(r + 8, rows)) for r in range(0, rows, 8)])
    for n in (40, 65, 300):
        got = product(0, n)
        assert torch.equal(got.isnan(), want[:n].isnan())
        clean = ~got.isnan()
        assert torch.equal(got[clean].view(torch.int32), want[:n][clean].view(torch.int32))


# the fifth row of a batch over weights that end in the middle of a round of tiles; outputs whose stripes of tiles leave places of a die empty
@pytest.mark.parametrize("width,count,rows,more,most", [(1024, 28672, 4, 5, 1.35), (3072, 12288, 4, 5, 1.35), (2048, (2048, 2195), 427, 427, 1.5)])
def test_a_little_more_costs_little(strix, width, count, rows, more, most):
    """No step from one round of the compute units to two, nearly twice the time, where another form takes less."""
    counts = count if isinstance(count, tuple) else (count, count)
    w = [strix.quantize_weight_rows(strix.TYPE_Q8_0, torch.randn((counts[1], width), device="cuda") * 0.02) for _ in range(8)]

    def micros(rows, count):
        codes, deltas, _, _ = strix.quantize_a8(torch.randn((rows, width), device="cuda"))
        y = torch.empty((rows, count), device="cuda")
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        taken = []
        for _ in range(7):
            torch.cuda.synchronize()
            begin.record()
            for i in range(64):
                strix.gemv_q8_0_a8(w[i % 8], codes, deltas, width, count, y)
            end.record()
            torch.cuda.synchronize()
            taken.append(begin.elapsed_time(end) * 1e3 / 64)
        return min(taken)

    before, after = micros(rows, counts[0]), micros(more, counts[1])
    assert after < most * before, (before, after)
