"""What the sweeps of contiguous Q4_K stages wait for, in the code that the compiler makes of them: a stage's LDS reads must not await the copies of the
next one, which were asked for in front of them."""
import os
import re
import shutil
import subprocess

import pytest

import __graft_entry__ as entry

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs the HIP compiler")

SOURCE = """
#include "q4k_blocks.hpp"
using namespace strix950;
template <int B> __global__ __launch_bounds__(512) void flat(const uint8_t* rows, A8Image image, float* out) {
    __shared__ __attribute__((aligned(16))) uint8_t even[8][kFlatStageBytes];
    __shared__ __attribute__((aligned(16))) uint8_t odd[8][kFlatStageBytes];
    __shared__ __attribute__((aligned(16))) uint8_t act[8][flat_act_bytes(B)];
    const uint32_t wave = threadIdx.x >> 6;
    lds_u8* const slots[2] = {(lds_u8*)even[wave], (lds_u8*)odd[wave]};
    image.table = nullptr;
    image.per_row = 1U;
    out[threadIdx.x] = sweep_flat_rows<B, 2>(slots, (lds_u8*)act[wave], rows, image, blockIdx.x);
}
template <int STAGES> __global__ __launch_bounds__(64) void terms(const uint8_t* rows, A8Image image, float* out) {
    __shared__ __attribute__((aligned(16))) uint8_t even[kFlatStageBytes];
    __shared__ __attribute__((aligned(16))) uint8_t odd[kFlatStageBytes];
    lds_u8* const slots[2] = {(lds_u8*)even, (lds_u8*)odd};
    image.table = nullptr;
    image.per_row = 1U;
    out[threadIdx.x] = sweep_block_lanes_terms<STAGES>(slots, [&](uint32_t s) { return rows + 9216U * s; }, block_lanes(STAGES, 32U), image, blockIdx.x);
}
template __global__ void flat<2>(const uint8_t*, A8Image, float*);
template __global__ void flat<3>(const uint8_t*, A8Image, float*);
template __global__ void flat<4>(const uint8_t*, A8Image, float*);
template __global__ void terms<4>(const uint8_t*, A8Image, float*);
template __global__ void terms<8>(const uint8_t*, A8Image, float*);
"""


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    where = tmp_path_factory.mktemp("sweeps")
    (where / "sweeps.hip").write_text(SOURCE)
    flags = [f for f in entry.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run(["hipcc"] + flags + ["-I" + os.path.join(entry.ROOT, "include"), "-I" + os.path.join(entry.PKG_DIR, "csrc"), "--cuda-device-only", "-S",
                    str(where / "sweeps.hip"), "-o", str(where / "sweeps.s")], check=True, stderr=subprocess.DEVNULL)
    return (where / "sweeps.s").read_text()


@pytest.mark.parametrize("kernel", ["flat<2>", "flat<3>", "flat<4>", "terms<4>", "terms<8>"])
def test_reads_do_not_await_the_next_stage(listing, kernel):
    name, number = re.fullmatch(r"(\w+)<(\d)>", kernel).groups()
    body = re.search(rf"^_Z\d+{name}ILi{number}E\S*:.*?s_endpgm", listing, re.S | re.M).group()
    found = re.findall(r"^\s*(global_load_lds_dword|s_waitcnt[^\n]*vmcnt\(0\)|ds_read_b128)", body, re.M)
    order = ["copy" if f.startswith("global") else "read" if f.startswith("ds") else "all" for f in found]
    steps = [o for i, o in enumerate(order) if i == 0 or o != order[i - 1]]
    assert steps.count("copy") >= 2 and "read" in steps
    # (the wait for a stage is followed by the next stage's copies, the last one by reads behind reads)
    assert not any(steps[i:i + 3] == ["copy", "all", "read"] for i in range(len(steps))), steps
