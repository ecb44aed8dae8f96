"""The GEMM's launch rules (csrc/gemm_plan.h) on the CPU, over their whole range.

The header is plain C++; a small program compiled here walks what the kernels would walk. No GPU."""

import pathlib
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
CSRC = ROOT / "vllm-omni-neuron_amd" / "csrc"


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """Compiles a C++ main that includes gemm_plan.h and returns what it prints."""

    def go(name: str, body: str) -> str:
        d = tmp_path_factory.mktemp(name)
        (d / "main.cc").write_text('#include "gemm_plan.h"\n#include <cstdio>\n#include <vector>\n'
                                   "using namespace wanmi;\n" + body)
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{CSRC}", str(d / "main.cc"),
                        "-o", str(d / "main")], check=True)
        return subprocess.run([str(d / "main")], check=True, capture_output=True, text=True, timeout=300).stdout

    return go


# Q|K and V widths: one and two weights of the model's 5120, grouped K/V heads (V narrow against Q|K), V wider
QKV_SWEEP = r"""
struct Width { int64_t qk, v; };
static const Width kWidths[] = {{10240, 5120}, {5120, 5120}, {6144, 1024}, {5120, 1024}, {5120, 512}, {5120, 256},
                                {10240, 2560}, {10240, 256}, {256, 256}, {256, 5120}, {1024, 10240}, {768, 512}};
template <class F>
void sweep(F f) {
  for (const Width& w : kWidths)
    for (int64_t cus : {256, 304, 128, 64, 38, 8, 2})
      for (int64_t M = 1; M <= 33000; M += M < 4200 && cus == 256 ? 1 : 61) {
        const int64_t vt_ld = (M + 63) / 64 * 64;
        f(M, w.qk, w.v, cus, select_qkv_tile(M, w.qk, w.v, cus, vt_ld));
      }
}
"""


def test_qkv_launch_has_a_tile_for_every_workgroup(run):
    """Q|K and V in one launch: both parts get a workgroup, and neither more workgroups than it has tiles (a
    workgroup without a tile of its own would compute one past the end of the weight and of V^T)."""
    out = run("qkv", QKV_SWEEP + r"""
int main() {
  long checked = 0, bad = 0;
  sweep([&](int64_t M, int64_t qk, int64_t v, int64_t cus, const TilePlan& p) {
    if (p.nj == 0 || p.cost == INT64_MAX) return;
    const int64_t mt = ceil_div(M, 64 * p.nj), tq = mt * (qk / TN), tv = mt * (v / TN);
    const int64_t v_wgs = tile_workgroups(p, tq + tv, cus) - p.qk_wgs;
    const int64_t rounds = std::max(ceil_div(tq, std::max<int64_t>(p.qk_wgs, 1)), ceil_div(tv, std::max<int64_t>(v_wgs, 1)));
    ++checked;
    if (p.qk_wgs < 1 || p.qk_wgs > tq || v_wgs < 1 || v_wgs > tv || p.qk_wgs + v_wgs > cus || p.cost != kTileCost[p.nj] * rounds) {
      if (bad++ < 5)
        printf("M=%ld qk=%ld v=%ld cus=%ld: nj=%d, %d workgroups for %ld tiles, %ld for %ld\n", (long)M, (long)qk, (long)v,
               (long)cus, p.nj, p.qk_wgs, (long)tq, (long)v_wgs, (long)tv);
    }
  });
  printf("checked %ld bad %ld\n", checked, bad);
}
""")
    assert out.splitlines()[-1].startswith("checked ") and out.endswith(" bad 0\n"), out


def test_run_panels_name_every_panel_a_run_reads(run):
    """The n tiles that an XCD's run of tiles reads, exactly, and token rows that hold all it reads, for every
    grid of at most 304 tiles (products of one round) of each tile that is fetched ahead of."""
    out = run("panels", r"""
static long checked, bad;
template <int kTm, int kGroup>
void grids() {
  for (int tm = 1; tm <= 304; ++tm)
    for (int tn = 1; tm * tn <= 304; ++tn)
      for (int64_t M : {(int64_t)(tm - 1) * kTm + 1, (int64_t)tm * kTm})
        for (int x = 0; x < 8; ++x) {
          const RunPanels p = run_panels<kTm, kGroup>(M, tm, tn, x);
          std::vector<int> want(tn, 0), got(tn, 0);
          bool rows = true;
          for (int v = x; v < tm * tn; v += 8) {
            const TileAt t = tile_at(v, tm, tn, kGroup);
            want[t.tn] = 1;
            rows &= (int64_t)t.tm * kTm >= p.m_lo && std::min<int64_t>((int64_t)(t.tm + 1) * kTm, M) <= p.m_hi;
          }
          bool inside = p.m_lo >= 0 && p.m_hi <= M && p.n0 + p.n_hi <= tn && p.n_lo <= tn;
          for (int i = 0; inside && i < p.n_hi; ++i) inside &= !got[p.n0 + i]++;
          for (int i = 0; inside && i < p.n_lo; ++i) inside &= !got[i]++;
          ++checked;
          if (!rows || !inside || want != got) {
            if (bad++ < 5) printf("%d x %d tiles of %d tokens, XCD %d: n [%d, +%d) and [0, %d)\n", tm, tn, kTm, x, p.n0, p.n_hi, p.n_lo);
          }
        }
}
int main() {
  grids<192, kGroupM * TM / 192>();
  grids<128, kGroupM * TM / 128>();
  grids<TS, kTsGroupM>();
  printf("checked %ld bad %ld\n", checked, bad);
}
""")
    assert out.splitlines()[-1].startswith("checked ") and out.endswith(" bad 0\n"), out


def test_qkv_split_is_that_of_the_search_over_all_splits(run):
    """Cost and tile as a search over every split of the CUs finds them, in well under a microsecond a call (the
    search took four)."""
    out = run("split", "#include <chrono>\n" + QKV_SWEEP + r"""
TilePlan search(int64_t M, int64_t qk, int64_t v, int64_t cus, int64_t vt_ld) {
  TilePlan best{4, INT64_MAX, 0};
  for (int nj : {4, 3, 2, 0}) {
    const int64_t tm = nj ? 64 * nj : TS, mt = ceil_div(M, tm);
    if (mt * tm < vt_ld) continue;
    if (nj == 0) {
      const int64_t cost = kTileCost[0] * ceil_div(mt * ((qk + v) / TS), cus);
      if (cost < best.cost) best = TilePlan{0, cost, 0};
      continue;
    }
    const int64_t tq = mt * (qk / TN), tv = mt * (v / TN);
    for (int64_t w = 1; w < std::min(cus, tq + tv); ++w) {
      const int64_t cost = kTileCost[nj] * std::max(ceil_div(tq, w), ceil_div(tv, std::min(cus, tq + tv) - w));
      if (cost < best.cost) best = TilePlan{nj, cost, (int)w};
    }
  }
  return best;
}
int main() {
  long checked = 0, bad = 0;
  sweep([&](int64_t M, int64_t qk, int64_t v, int64_t cus, const TilePlan& p) {
    const TilePlan want = search(M, qk, v, cus, (M + 63) / 64 * 64);
    ++checked;
    if (p.nj != want.nj || p.cost != want.cost) ++bad;
  });
  printf("checked %ld bad %ld\n", checked, bad);
  int64_t sum = 0;
  double best = 1e9;
  for (int rep = 0; rep < 5; ++rep) {
    const auto t0 = std::chrono::steady_clock::now();
    for (int64_t M = 1; M <= 20000; ++M) sum += select_qkv_tile(M, 10240, 5120, 256, (M + 63) / 64 * 64).cost;
    best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 20000);
  }
  printf("%lld\n%.3f\n", (long long)sum, best);
}
""").splitlines()
    assert out[0].startswith("checked ") and out[0].endswith(" bad 0"), out
    assert float(out[2]) < 1.0, f"{out[2]} us per call"
