"""What the compiler makes of the pipelined GEMM's prologue (CPU, the build's own assembly).

Between two tiles a workgroup clears its accumulators and nothing else may stand between the next tile's first
stage and its MFMAs. Clearing them twice (once for a k loop that never runs) costs about 0.5 us per tile."""

import importlib.util
import pathlib
import re

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
_spec = importlib.util.spec_from_file_location("wanmi_build", ROOT / "vllm-omni-neuron_amd" / "build.py")
build = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(build)


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    """Device assembly of mxfp8_gemm.hip: the last build's if it is newer than every source, else made here."""
    built = build.BUILD_DIR / "mxfp8_gemm.s"
    sources = [*build.CSRC.glob("*"), *build.INCLUDE_DIR.glob("*"), ROOT / "vllm-omni-neuron_amd" / "build.py"]
    if built.exists() and built.stat().st_mtime > max(s.stat().st_mtime for s in sources):
        return built.read_text()
    build.BUILD_DIR = tmp_path_factory.mktemp("asm")
    return build._device_asm(build.CSRC / "mxfp8_gemm.hip", [])


def test_accumulators_are_cleared_once_per_tile(asm):
    kernels = re.findall(r"^(_ZN5wanmi22mxfp8_gemm_ring_kernelILi(\d+)ELi(\d)EEE\w+):(.*?)^\.Lfunc_end", asm, re.M | re.S)
    assert len(kernels) == 18
    for name, epilogue, nj, body in kernels:
        if epilogue == "101":  # two tile loops, one after the other in the text
            continue
        before = body[: body.index("v_mfma")]
        clears = len(re.findall(r"v_accvgpr_write_b32 a\d+, 0\b(?!x)", before))
        # 64 accumulator registers per token fragment; a few more zeros are other operands
        assert clears <= 64 * int(nj) + 8, (name, clears)
