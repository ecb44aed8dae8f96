"""Spilled registers of the Q/K pass, as the compiler reports them for the flags of the build (CPU).

The single passes of up to 40 heads run at 128 registers per wave, so that four waves fit a SIMD; what one
needs beyond is spilled to memory in its token loop, and a few registers more cost up to a tenth of a long
pass. The bounds are what these kernels' own work needs (halves: eight angles per lane instead of four)."""

import importlib.util
import pathlib
import re
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
_spec = importlib.util.spec_from_file_location("wanmi_build", ROOT / "vllm-omni-neuron_amd" / "build.py")
build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(build)


@pytest.fixture(scope="module")
def spills(tmp_path_factory):
    """{(chunks, halves, out, pair): most VGPRs spilled over the workgroup sizes} of the built instantiations."""
    out = tmp_path_factory.mktemp("qk_prep") / "qk_prep.s"
    subprocess.run([build._hipcc(), *build.HIP_FLAGS, f"-I{build.INCLUDE_DIR}", "--cuda-device-only", "-S",
                    str(build.CSRC / "qk_prep.hip"), "-o", str(out)], check=True, capture_output=True)
    found = {}
    for name, n in re.findall(r"\.name:\s+(\S*qk_rmsnorm_rope_kernel\S*).*?\.vgpr_spill_count:\s+(\d+)", out.read_text(), re.S):
        chunks, halves, to, _, pair = re.search(r"ILi(\d+)ELb(\d)ELb(\d)ELi(\d+)(?:ELb(\d))?", name).groups()
        key = int(chunks), halves == "1", to == "1", pair == "1"
        found[key] = max(found.get(key, 0), int(n))
    assert found
    return found


def test_single_passes_spill_what_their_own_work_needs(spills):
    bound = {(10, False, False): 2, (10, True, False): 11, (10, False, True): 9, (10, True, True): 23}
    for (chunks, halves, out, pair), n in spills.items():
        if not pair and chunks <= 10:
            assert n <= bound.get((chunks, halves, out), 0), (chunks, halves, out, n)
    assert all((*k, False) in spills for k in bound)
