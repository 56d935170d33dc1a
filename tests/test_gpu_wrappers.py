"""The native wrappers (host/torch_ops.cpp) as Python callers see them: torch's own exception types come through."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def strix():
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


def product(strix, rows=3, width=64, count=5):
    w = strix.quantize_weight_rows(strix.TYPE_Q8_0, torch.randn((count, width), device="cuda"))
    codes, deltas, _, _ = strix.quantize_a8(torch.randn((rows, width), device="cuda"))
    return w, codes, deltas, width, count


def test_allocation_failure_is_out_of_memory(strix):
    rows = torch.zeros((1, 1 << 24), dtype=torch.float16, device="cuda").expand(65535, 1 << 24)       # an image of 1.1 TB
    with pytest.raises(torch.OutOfMemoryError):
        strix.quantize_a8(rows)


def test_shape_errors_keep_their_type(strix):
    w, codes, deltas, width, count = product(strix)
    with pytest.raises(IndexError):
        strix.gemv_q8_0_a8(w, codes[0], deltas, width, count)
    with pytest.raises(RuntimeError, match="ambiguous"):
        strix.gemv_q8_0_a8(w, codes, deltas, width, count, accumulate=torch.ones(2))
