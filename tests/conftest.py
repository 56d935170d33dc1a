import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def strix():
    """The GPU library binding. Fails loudly when the HIP extension is missing or no GPU is present."""
    from __graft_entry__ import load_package
    pkg = load_package()
    pkg.require_gpu()
    return pkg


class PrefillForm:
    """The workgroup form that the fp16 prefill is made to take, and a look at the plan for the one that a layer took."""
    FORMS = {"by_size": (0, None), "four_waves": (1, 32), "wide": (2, 128)}
    OFFSETS_AT = 2240                              # first word of the plan arrays (offsets, touched, order, items)

    def __init__(self, lib):
        self.lib = lib

    def use(self, name):
        self.name = name
        self.lib.mi355_debug_prefill_form(self.FORMS[name][0])

    def check(self, layer, name=None):
        pad4 = lambda n: (n + 3) // 4 * 4
        plan, experts = layer.plan.cpu().numpy(), layer.w.experts
        at = self.OFFSETS_AT + pad4(experts + 1) + pad4(experts) + pad4(int(plan[0]))
        items = plan[at:at + 4 * plan[4]].reshape(-1, 4)
        assert (items[:, 2] - items[:, 1]).max() == min(int(plan[2]), self.FORMS[name or self.name][1])


@pytest.fixture(params=["four_waves", "wide"])
def prefill_form(strix, request):
    form = PrefillForm(strix.lib())
    form.use(request.param)
    yield form
    form.use("by_size")


@pytest.fixture
def prefill_forms(strix):
    form = PrefillForm(strix.lib())
    yield form
    form.use("by_size")
