"""The native wrappers (host/torch_ops.cpp) as Python callers see them: torch's own exception types come through, and other threads
run during a call."""
import sys
import threading
import time

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


def test_other_threads_run_during_a_call(strix):
    """With a switch interval longer than the test only a call that gives the interpreter up lets the other thread in."""
    args = product(strix)
    x = torch.randn((3, 64), device="cuda")
    interval, turns, stop = sys.getswitchinterval(), [0], threading.Event()

    def count():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)

    for call in (lambda: strix.quantize_a8(x), lambda: strix.gemv_q8_0_a8(*args)):
        stop.clear()
        thread = threading.Thread(target=count)
        thread.start()
        try:
            sys.setswitchinterval(1000.0)
            time.sleep(0.05)                   # (a wait that the thread began before still ends after the old interval)
            before = turns[0]
            for _ in range(5000):
                call()
                if turns[0] != before:
                    break
            after = turns[0]
        finally:
            sys.setswitchinterval(interval)
            stop.set()
            thread.join()
        assert after > before
    torch.cuda.synchronize()


def test_operands_in_pinned_host_memory(strix):
    """The product reads and writes host memory that the GPU can reach; memory that it cannot is refused."""
    w, codes, deltas, width, count = product(strix)
    want = strix.gemv_q8_0_a8(w, codes, deltas, width, count)

    def pinned(t):
        host = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
        host.copy_(t)
        return host

    assert torch.equal(strix.gemv_q8_0_a8(pinned(w), codes, pinned(deltas), width, count), want)
    out = pinned(torch.zeros_like(want))
    strix.gemv_q8_0_a8(pinned(w), pinned(codes), deltas, width, count, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out, want.cpu())
    for bad in ((w.cpu(), codes, deltas), (w, codes.cpu(), deltas), (w, codes, deltas.cpu()), (w, pinned(codes), deltas)):
        with pytest.raises(RuntimeError, match="GPU"):      # (the last has nowhere to put its output)
            strix.gemv_q8_0_a8(*bad, width, count)
    with pytest.raises(RuntimeError, match="GPU"):
        strix.gemv_q8_0_a8(w, codes, deltas, width, count, out=want.cpu())
