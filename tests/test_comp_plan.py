"""The host-side choices of a closed-set plan (quac_amd/csrc/qh_comp_plan.h), compiled
with the host compiler: every launch that a plan can hold has a kernel whose thread
count, rows a thread, slots and LDS take every bin of the launch, and every bin is in
one launch."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "quac_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """run(name, body): body's output, compiled behind the header with a main()"""
    d = tmp_path_factory.mktemp("plan")

    def _run(name, body):
        src, exe = str(d / (name + ".cpp")), str(d / name)
        heads = ["<array>", "<cstdio>", "<cstdlib>", "<random>", '"qh_comp_plan.h"', '"qh_optional.h"']
        with open(src, "w") as f:
            f.write("".join(f"#include {h}\n" for h in heads) + body)
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined", "-I", CSRC, src,
                        "-o", exe], check=True)
        return subprocess.run([exe], check=True, capture_output=True, text=True).stdout

    return _run


CHECK = r"""
#define NEED(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); exit(1); } } while (0)
[[maybe_unused]] static const int CUS = 256;
static void walk(const std::vector<CpBin> &bin, bool f32, const CpShapes &s, const std::vector<CpClass> &classes) {
  std::vector<int> seen(bin.size());
  int at = 0;
  for (const CpClass &k : classes) {
    NEED(k.first == at && k.count > 0 && cp_has_kernel(k));
    NEED(k.threads <= 1024 && k.threads % 64 == 0);
    // two buffers of k.cells entries, and the table beside words
    const size_t cell = k.W == 0 && f32 ? 8 : 16;
    NEED(2 * cell * k.cells + (k.W == 0 ? 8 * CP_DICT : 0) <= 160 * 1024);
    for (int i = 0; i < k.count; i++) {
      const CpBin &b = bin[s.bins[at + i]];
      seen[s.bins[at + i]]++;
      NEED(s.words[s.bins[at + i]] == (k.W == 0));
      NEED(b.rows <= k.threads * k.S && b.rows + 1 <= k.cells);
      if (k.W) NEED(b.width <= k.W);
    }
    at += k.count;
  }
  NEED(at == (int)bin.size());
  for (int n : seen) NEED(n == 1);
  NEED(!classes.back().side);
}
[[maybe_unused]] static void check(const std::vector<CpBin> &bin, bool f32) {
  const CpShapes s = cp_shapes(bin, f32, CUS);
  NEED(s.runnable);
  walk(bin, f32, s, s.classes);
  NEED(s.brief.empty() ? s.brief_steps == 0 : s.brief_steps >= 0 && s.brief.size() < s.classes.size());
  if (!s.brief.empty()) walk(bin, f32, s, s.brief);
  for (const CpClass &k : s.brief) NEED(!k.side);
}
"""


def test_every_launch_has_a_kernel(run):
    out = run("shapes", CHECK + r"""
int main() {
  // every pair of bins: up to one slice, up to one and two rows a thread, and words,
  // beside every width of a slice
  const int rows[] = {64, 128, 192, 512, 576, 1024, 1088, 2048, 2112, 4800};
  const int widths[] = {0, 4, 5, 8, 9, 10, 11, 12, 13, 16, 24, 32, 33};
  for (int few = 0; few < 2; few++)
    for (int r1 : rows)
      for (int r2 : rows)
        for (int w1 : widths)
          for (int w2 : widths) {
            std::vector<CpBin> bin{{r1, w1, (int64_t)w1 * r1 / 64}, {r2, w2, (int64_t)w2 * r2 / 64}};
            if (!few) bin.resize(2 * CUS + 1, bin[0]);
            check(bin, (w1 + w2) & 1);
          }
  std::mt19937 rng(7);
  for (int t = 0; t < 1000; t++) {
    std::vector<CpBin> bin(1 + rng() % (t % 8 ? 24 : 900));
    for (CpBin &b : bin) {
      b.rows = 64 * (1 + rng() % (rng() % 4 ? 16 : 75));
      b.width = rng() % (rng() % 3 ? 14 : 40);
      b.slots = (int64_t)b.width * (b.rows / 64);
    }
    check(bin, t & 1);
  }
  printf("ok\n");
}
""")
    assert out == "ok\n"


def test_short_calls_take_fewer_launches(run):
    """many small bins go into one launch for a call of few steps, whatever the steps of
    a larger one; bins of a launch of their own stay in it where the rest would idle"""
    out = run("brief", CHECK + r"""
static std::vector<CpBin> bins(std::vector<std::array<int, 3>> groups) {
  std::vector<CpBin> b;
  for (auto g : groups)
    for (int i = 0; i < g[0]; i++) b.push_back({g[1], g[2], (int64_t)g[2] * g[1] / 64});
  return b;
}
int main() {
  // the bins of decay and dephasing of 8, 10 and 11 qubits
  const auto b8 = bins({{9, 256, 8}, {233, 128, 7}, {128, 128, 4}, {266, 64, 6}, {369, 64, 4}});
  const auto b10 = bins({{9, 1024, 10}, {12, 512, 9}, {2156, 512, 7}, {16, 512, 4}, {9, 64, 4}});
  const auto b11 = bins(
      {{9, 2048, 11}, {102, 1024, 10}, {132, 512, 9}, {8458, 512, 8}, {22, 512, 4}, {57, 256, 8}, {13, 64, 8}});
  const CpShapes s8 = cp_shapes(b8, false, CUS), s10 = cp_shapes(b10, false, CUS), s11 = cp_shapes(b11, false, CUS);
  NEED(s8.classes.size() == 5 && s8.brief.size() == 1 && s8.brief_steps >= 20);
  NEED(s10.brief.size() == 1 && s10.brief_steps >= 2 && s10.brief_steps <= 20);
  NEED(s11.brief.size() == 1 && s11.brief_steps == 0);
  printf("ok\n");
}
""")
    assert out == "ok\n"


def test_plan_waits_for_the_steps_that_pay_for_it(run):
    """few steps never wait for a plan, a graph's worth of them on a small matrix does,
    and steps in several calls count together"""
    out = run("pays", CHECK + r"""
int main() {
  for (int64_t n : {801, 1296, 4096, 8464, 16384, 16385, 57600, 65536}) {
    NEED(!cp_pays(n, 0, 0, 8, true) && !cp_pays(n, 0, 1, 8, true) && !cp_pays(n, 0, 4, 8, true));
    NEED(cp_pays(n, 0, 20, 8, true) && cp_pays(n, 0, 100, 8, true));
    int64_t k = 0;
    while (!cp_pays(n, k, 1, 8, true)) k++;
    NEED(k >= 4 && k <= 40);
    NEED(!cp_pays(n, 0, k, 1000, true) && cp_pays(n, 0, k + 1, 1000, true));
    for (int64_t s = 1; s < 100; s++) NEED(cp_pays(n, s, 5, 8, true) || !cp_pays(n, s - 1, 5, 8, true));
    NEED(!cp_pays(n, 3, 2, 8, true) || cp_pays(n, 3, 2, 8, false));
  }
  // 16 M rows: ten steps with the layout still to be built
  NEED(cp_pays(16777216, 0, 10, 8, false) && !cp_pays(16777216, 0, 10, 8, true));
  printf("ok\n");
}
""")
    assert out == "ok\n"


def test_side_stream_is_joined_when_a_launch_fails(run):
    """the order of fork, launches and join for every launch that may fail"""
    out = run("order", CHECK + r"""
int main() {
  for (int sides = 0; sides < 2; sides++)
    for (int bad = -1; bad < 4; bad++) {
      std::vector<CpClass> c(4, CpClass{64, 1, 4, true, false, 0, 1, 65});
      c[0].side = c[2].side = sides;
      int forks = 0, joins = 0, launched = 0;
      const int rc = cp_run(
          c,
          [&](const CpClass &k) {
            NEED(!k.side || (forks == 1 && joins == 0));
            return launched++ == bad ? -7 : 0;
          },
          [&] { return forks++, 0; }, [&] { return joins++, 0; });
      NEED(rc == (bad < 0 ? 0 : -7) && launched == (bad < 0 ? 4 : bad + 1));
      NEED(forks == sides && joins == sides);
      NEED(cp_run(c, [](const CpClass &) { return 0; }, [] { return 0; }, [] { return -3; }) == (sides ? -3 : 0));
      int n = 0;
      NEED(cp_run(c, [&](const CpClass &) { return n++, 0; }, [] { return -5; }, [&] { return n++, 0; }) ==
           (sides ? -5 : 0) && n == (sides ? 0 : 4));
    }
  printf("ok\n");
}
""")
    assert out == "ok\n"


def test_no_memory_for_a_plan_is_no_error(run):
    """a plan or list that does not fit in memory is done without; other errors stay"""
    out = run("optional", CHECK + r"""
int main() {
  int none = 0;
  auto n = [&] { none++; };
  NEED(qh_optional(-2, [] { return 0; }, n) == 0 && none == 0);
  NEED(qh_optional(-2, [] { return -3; }, n) == -3 && none == 0);
  NEED(qh_optional(-2, [] { return -2; }, n) == 0 && none == 1);
  NEED(qh_optional(-2, []() -> int { throw std::bad_alloc(); }, n) == 0 && none == 2);
  printf("ok\n");
}
""")
    assert out == "ok\n"
