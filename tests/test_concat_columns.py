"""The columns a workgroup of the concat kernel takes: few threads without an element, and chosen in no time a caller
of a small concatenation would notice (a whole call is some 4 us of host time)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flexflow-train_amd", "csrc")
PROGRAM = r"""
#include "concat_columns.h"
#include <algorithm>
#include <chrono>
#include <cstdio>
int main() {
  for (long units = 1; units <= 5000; units++)
    for (long rows : {1l, 2l, 3l, 100l, 1000000l}) printf("%ld %ld %d\n", units, rows, ffk::concat_columns(units, rows));
  printf("%ld %ld %d\n", 1l << 40, 1l << 30, ffk::concat_columns(1l << 40, 1l << 30));
  double least = 1e9;
  for (int turn = 0; turn < 20; turn++) {
    volatile int sum = 0;
    auto const t = std::chrono::steady_clock::now();
    for (int i = 0; i < 10000; i++) sum = sum + ffk::concat_columns(150 + i % 400, 1000);
    least = std::min(least, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t).count() / 10000);
  }
  fprintf(stderr, "%f\n", least);
}
"""


def test_columns_of_a_workgroup(tmp_path):
    (tmp_path / "t.cc").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(tmp_path / "t.cc"), "-o", str(tmp_path / "t")], check=True)
    run = subprocess.run([str(tmp_path / "t")], check=True, capture_output=True, text=True)

    def busy(units, rows, cols):  # share of a launch's threads with an element
        return units * min(256 // cols, rows) / (256 * -(-units // cols))

    for line in run.stdout.splitlines():
        units, rows, cols = map(int, line.split())
        assert 1 <= cols <= min(units, 256), line
        share = busy(units, rows, cols)
        # never worse than as many columns as there are, nor, with rows in plenty, a tenth behind the best width
        assert share >= busy(units, rows, min(units, 256)), line
        if rows == 1000000 and units <= 300:
            assert share >= 0.9 * max(busy(units, rows, c) for c in range(1, min(units, 256) + 1)), line
    assert float(run.stderr) < 0.5, "microseconds a choice: " + run.stderr
