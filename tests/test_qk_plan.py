"""The Q/K pass's launch rule (csrc/qk_plan.h) on the CPU, over its whole range. No GPU."""

import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "vllm-omni-neuron_amd" / "csrc"


def _run(d, body):
    """What a C++ main over qk_plan.h prints: a tuple of numbers per line."""
    (d / "main.cc").write_text('#include "qk_plan.h"\n#include <cstdio>\n#include <initializer_list>\n' + body)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{CSRC}", str(d / "main.cc"), "-o",
                    str(d / "main")], check=True)
    out = subprocess.run([str(d / "main")], check=True, capture_output=True, text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    """[(heads, rows, maxnorm, cus, chunks, waves, tokens per wave)]"""
    return _run(tmp_path_factory.mktemp("qk_plan"), r"""
int main() {
  for (int heads = 4; heads <= 128; heads += 4)
    for (long rows : {1l, 512l, 4096l, 4097l, 28672l, 28673l, 32760l, 75600l, 1l << 31})
      for (int max : {0, 1})
        for (int cus : {32, 256}) {
          const wanmi::QKPlan p = wanmi::qk_plan(heads, rows, max != 0, cus);
          printf("%d %ld %d %d %d %d %d\n", heads, rows, max, cus, p.chunks, p.waves, p.tokens_per_wave);
        }
}
""")


def test_every_pass_takes_the_smallest_instantiation_that_holds_its_heads(plans):
    for heads, rows, maxnorm, cus, chunks, waves, _ in plans:
        assert chunks == min(c for c in (4, 10, 16, 32) if 4 * c >= heads), (heads, maxnorm)
        assert waves in (4, 8) and (waves == 4 or (maxnorm and heads <= 40))


def test_a_resident_round_of_waves_comes_before_a_second_token(plans):
    for heads, rows, maxnorm, cus, _, _, tokens in plans:
        assert 1 <= tokens <= 8 and (tokens == 8 or tokens * cus * 16 >= rows)
        assert tokens == 1 or (tokens - 1) * cus * 16 < rows


def test_long_passes_end_in_workgroups_of_four_waves(plans):
    """With every wave at its most tokens the pass is bound by memory, and larger workgroups only lengthen its
    end; up to 8 heads the maxima's atomics still bound it."""
    for heads, rows, maxnorm, cus, _, waves, tokens in plans:
        if maxnorm and heads <= 40:
            assert waves == (4 if tokens == 8 and heads > 8 else 8), (heads, rows, cus)


def test_the_maximum_alone_takes_large_workgroups_only_where_atomics_bound_it(tmp_path):
    """Eight waves per workgroup neither over a few hundred tokens nor over more than memory streams anyway."""
    faster = {(64, 4): 4, (256, 40): 4, (512, 24): 4, (1024, 40): 8, (2500, 4): 8, (7800, 40): 8, (32760, 24): 8,
              (32760, 40): 4, (50000, 32): 4, (75600, 40): 4}  # (tokens, heads): as measured
    calls = "".join(f'printf("%d\\n", wanmi::head_max_norm_waves({r}, {h}));' for r, h in faster)
    assert [w for w, in _run(tmp_path, "int main() {" + calls + "}")] == list(faster.values())
