"""Registers and LDS of the built kernels, from the code objects' metadata."""
import os
import re
import subprocess

import pytest

from wind_amd import api

LLVM = "/opt/rocm/llvm/bin"
pytestmark = pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-readelf"), reason="needs the ROCm LLVM tools")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> (VGPRs, declared LDS bytes) of the core library."""
    d = tmp_path_factory.mktemp("co")
    os.symlink(api.LIB_PATH, d / "lib.so")
    subprocess.run([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    out = {}
    for co in (f for f in os.listdir(d) if "gfx950" in f):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", co], cwd=d, check=True, capture_output=True,
                               text=True).stdout
        for k in notes.split("- .agpr_count:")[1:]:
            get = lambda key: re.search(rf"\.{key}:\s+(\S+)", k).group(1)
            name = subprocess.run(["c++filt", get("name")], check=True, capture_output=True, text=True).stdout
            out[name.strip()] = (int(get("vgpr_count")), int(get("group_segment_fixed_size")))
    return out


def find(kernels, text):
    got = [v for k, v in kernels.items() if text in k]
    assert len(got) == 1, (text, got)
    return got[0]


@pytest.mark.parametrize("kernel", ["NRTest, 1, false", "Katz96, 1, false", "Katz96, 1, true", "HHe6, 1, false",
                                    "HHe6, 1, true"])
def test_explicit_row_kernels_declare_no_lds(kernels, kernel):
    """Nothing of theirs is indexed per thread: arrays that the compiler moves to LDS for that cost every launch a
    read of its packet in host memory."""
    assert find(kernels, f"row_integrate<wind::Net{kernel}>")[1] == 0


@pytest.mark.parametrize("net", ["Katz96", "HHe6"])
@pytest.mark.parametrize("method", [0, 1])
def test_hand_over_leaves_the_lane_kernels_their_waves(kernels, net, method):
    """As many waves per SIMD (512 VGPRs, given in eights) with the hand-over in the loop as without it."""
    waves = [512 // (-(-find(kernels, f"lane_integrate<wind::Net{net}, {method}, wind::MathExact, false, {spill}>")[0]
                       // 8) * 8) for spill in (0, 1)]
    assert waves[0] == waves[1]
