"""What the built kernels take of the register file, where their time depends on it. Runs without a GPU."""
import re
import subprocess

import pytest

from tests.test_wait_states import code_object


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel name: (VGPRs, spilled SGPRs, spilled VGPRs)} from the code object's notes."""
    co, tool = code_object(tmp_path_factory.mktemp("co"))
    notes = subprocess.run([tool("llvm-readelf"), "--notes", co], check=True, capture_output=True, text=True).stdout
    out = {}
    for part in notes.split(".args:")[1:]:
        name = re.findall(r"\.name:\s+(_Z\S+)", part)
        if name:
            plain = subprocess.run(["c++filt", name[0]], check=True, capture_output=True, text=True).stdout
            plain = plain.replace("(anonymous namespace)::", "").replace("void ", "").split("(")[0].strip()
            out[plain] = tuple(int(re.search(rf"\.{k}:\s+(\d+)", part).group(1)) for k in ("vgpr_count", "sgpr_spill_count", "vgpr_spill_count"))
    return out


@pytest.mark.parametrize("Q", [1024, 2048, 4096])
def test_packed_replay(kernels, Q):
    """The replay-only kernel of the packed form keeps its scalars (each spilled one is a lane read in a loop over copies)
    and the waves its LDS allows; the kernel with the decoder does not spill hundreds for the sake of the packed form.
    Bounds: 64 VGPRs are eight waves per SIMD, twice what the LDS lets in; with 2 spilled SGPRs the replay of 65,536 windows
    takes as long as with none (417 us), with 135 it took 426."""
    vgpr, sgpr_spill, vgpr_spill = kernels[f"windows_kernel<{Q}, false, false, false>"]
    assert vgpr <= 64 and sgpr_spill <= 16 and vgpr_spill == 0
    assert kernels[f"windows_kernel<{Q}, true, false, false>"][1] <= 256


@pytest.mark.parametrize("Q", [1024, 2048, 4096])
def test_front_kernel_four_waves(kernels, Q):
    """front_kernel decodes each long block by a wave of its own: 128 VGPRs, four waves per SIMD."""
    vgpr, _, vgpr_spill = kernels[f"front_kernel<{Q}, false>"]
    assert vgpr <= 128 and vgpr_spill <= 4
