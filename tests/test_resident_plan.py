"""The plan of the resident-key kernel (csrc/resident_plan.h), compiled for the CPU: the search that prices few numbers of workgroups finds what
pricing all of them finds."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "resident_plan.h"
using namespace pa;
int main() {
  int wrong = 0, most_priced = 0;
  const int cu_counts[] = {256, 304, 80, 1};
  const int heads[] = {1, 2, 3, 7, 12, 24, 25, 40, 48, 64, 80, 100, 128, 255, 256, 257, 300, 513, 1000, 5000};
  for (int cus : cu_counts)
    for (int h : heads)
      for (int n = 1; n <= 8192; n += n < 1100 ? 1 : 97) {
        int best = 1;
        double best_cost = 1e30;
        for (int parts = 1; parts <= (n + 3) / 4 && parts <= 4 * cus; ++parts) {
          const double cost = resident_cost(h, n, cus, parts);
          if (cost < best_cost * 0.999) {
            best_cost = cost;
            best = parts;
          }
        }
        int priced = 0;
        const int got = resident_parts(h, n, cus, &priced);
        if (got != best && wrong++ < 10) printf("%d units of %d heads on %d: %d, all priced %d\n", n, h, cus, got, best);
        if (priced > most_priced) most_priced = priced;
      }
  int a = 0, b = 0;
  resident_parts(24, 1024, 256, &a);
  resident_parts(24, 4096, 256, &b);
  printf("wrong %d most %d 24x1024 %d 24x4096 %d\n", wrong, most_priced, a, b);
  return wrong != 0;
}
"""


def test_search_equals_pricing_every_number(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "paraattention_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout
    most = int(run.stdout.split("most ")[1].split()[0])
    assert most <= 160, run.stdout  # prices of one plan, of up to 1024
