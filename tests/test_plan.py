"""Launch rules of fk_plan.h on the host: what a launch writes fits the buffer
that was sized for it, and grids hold the lanes that their kernels use."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    """Compiles main's body against fk_plan.h and returns its output lines."""
    d = tmp_path_factory.mktemp("plan")

    def run(body):
        src, exe = d / "probe.cpp", d / "probe"
        src.write_text('#include <cstdio>\n#include <vector>\n#include "fk_plan.h"\nusing namespace fkx;\n'
                       'int main() {\n' + body + '\n  return 0;\n}\n')
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unused-function", "-Wno-parentheses",
                        "-I" + os.path.join(ROOT, "fooskagpu_amd", "csrc"), str(src), "-o", str(exe)], check=True)
        return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")[:-1]

    return run


def test_relaxation_counts_fit_their_buffer_at_either_precision(probe):
    """The buffer of the partial counts is sized once a mesh, the precision and
    the kind of relaxation may change after that: the words of every launch
    (blocks of the relaxation's own kernels, waves of a pass F that relaxes)
    at either precision, around each size where a rule changes and up to the
    largest mesh."""
    lines = probe("""
  std::vector<int64_t> sizes;
  for (int64_t n = 1; n < 2000; ++n) sizes.push_back(n);
  for (int64_t at : {22000, 25000, 30000, 35000, 50000, 60000, 120000, 160000, 220000, 350000, 600000})
    for (int64_t d = -300; d <= 300; ++d) sizes.push_back(at + d);
  for (int64_t n = 2000; n < (int64_t)1 << 28; n += n / 7) sizes.push_back(n);
  long tried = 0;
  for (int ns : {4, 6})
    for (int64_t nc : sizes) {
      const int64_t cap = relax_words(nc, ns);
      int64_t most = (int64_t)grid_for(nc) * 4;
      for (int relax = 1; relax <= 2; ++relax)
        for (int f64 = 0; f64 <= 1; ++f64) {
          for (int block : {128, 256}) most = std::max(most, pass_f_waves(nc, block) * (1 + relax));
          if (nc <= quad_cells_f(f64, ns, 10, relax)) most = std::max(most, (int64_t)grid_quad(nc) * (1 + relax));
        }
      ++tried;
      if (most > cap) std::printf("%d slots, %ld cells: %ld words of %ld\\n", ns, (long)nc, (long)most, (long)cap);
    }
  std::printf("tried %ld\\n", tried);""")
    assert lines[:-1] == [] and int(lines[-1].split()[1]) > 10000, lines[:5]


def test_a_list_takes_few_rounds_on_groups(probe):
    """Listed cells on groups of lanes (8 a chemical solve, 4 a polish): a list
    that takes groups needs at most four rounds of the grid (two of a polish),
    up to 65,536 (49,152) cells of any mesh the list does take them, and one
    lane a cell needs one round up to 262,144 cells."""
    lines = probe("""
  auto rounds = [](int64_t lanes, int64_t nt) { return (lanes + nt - 1) / nt; };
  for (int64_t nc = 1; nc <= 1 << 20; nc += 1 + nc / 50)
    for (int64_t n = 1; n <= nc; n += 1 + n / 20) {
      const int64_t nt8 = (int64_t)list_blocks(nc, 8) * kBlock, nt4 = (int64_t)list_blocks(nc, 4) * kBlock;
      const int l8 = chem_lanes(n, nt8), l4 = polish_lanes(n, nt4), lf = chem_lanes(n, std::min<int64_t>(nt8, 512 * kBlock));
      if (l8 != (n <= kChemGroup ? 8 : 1) || l4 != (n <= kPolishGroup ? 4 : 1) || lf != l8 || rounds(n * 8, nt8) > 4 && l8 == 8 ||
          rounds(n * 4, nt4) > 2 && l4 == 4 || n <= 262144 && (rounds(n, nt8) > 1 || rounds(n, nt4) > 1))
        std::printf("%ld of %ld cells: %d %d\\n", (long)n, (long)nc, l8, l4);
    }
  std::printf("%u %u %u\\n", list_blocks(1, 8), list_blocks(20000, 8), list_blocks((int64_t)1 << 30, 8));""")
    assert lines == ["1 512 1024"], lines[:5]
