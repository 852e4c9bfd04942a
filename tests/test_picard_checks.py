"""The rule for the Picard loop's separate residual tests (frehg_amd/csrc/picard_checks.hpp), compiled for the host:
an iterate that failed its test is not tested in the next step, and is tested again once a loop has ended there
or before, so that one hard step does not keep later ones from the cheaper path."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "picard_checks.hpp"

// A step whose iterates h^1 .. h^(n-1) fail their residual test and whose loop ends at h^n; returns the iterates
// that were tested (a test of h^n passes; an untested one ends by the increment or by its solve).
static std::vector<int> step(frehg::PicardChecks& c, int n) {
  std::vector<int> tested;
  for (int m = 1;; ++m) {
    const bool test = !c.expect_fail(m);
    if (test) tested.push_back(m);
    if (m == n) {
      c.ended(m);
      return tested;
    }
    if (test) c.failed(m);
  }
}

int main() {
  frehg::PicardChecks c;
  for (int n : {1, 3, 3, 3, 2, 2, 2, 1, 1, 3, 40, 40, 35, 1, 1}) {
    for (int m : step(c, n)) std::printf("%d ", m);
    std::printf("\n");
  }
  step(c, 5);
  c.clear();
  for (int m : step(c, 3)) std::printf("%d ", m);
  std::printf("\n");
  return 0;
}
"""


def test_which_iterates_are_tested(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "frehg_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines()
    got = [[int(v) for v in line.split()] for line in out]
    late = list(range(32, 41))  # beyond the 31 iterates that are remembered: always tested
    assert got[:10] == [[1],
                        [1, 2, 3],  # a storm step: two tests fail
                        [3], [3],  # ... and are left out while they would fail again
                        [],  # ends at h^2, which was expected to fail
                        [2], [2],  # tested again from the next step on
                        [],  # ends at h^1
                        [1],  # tested again
                        [1, 2, 3]]  # nothing is remembered of iterates that a step did not reach
    assert got[10] == list(range(3, 41)) and got[11] == late
    assert got[12] == list(range(32, 36)) and got[13] == [] and got[14] == [1]
    assert got[15] == [1, 2, 3]
