"""The cooperative tridiagonalisation's exchange (coop_exchange.hpp), on the
CPU: workers that run as far ahead of one another as the words allow must
never find a word of theirs overwritten. Compiled from the kernels' own rule."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "baandi_amd", "csrc")

SOURCE = r"""
#include "coop_exchange.hpp"
#include <cstdio>
#include <vector>
// One worker (`late`) runs only when no other can. Every worker at step k
// publishes its exchanged words into slot k % 2, then waits until all the
// exchanged words of its step are there. A word is its tag, k + 1.
static bool finishes(int m, int nw, int late) {
  std::vector<std::vector<int>> slot(2, std::vector<int>(m, 0));
  std::vector<int> step(nw, 0);
  std::vector<char> sent(nw, 0);
  const int steps = m - 2;
  auto advance = [&](int w) {
    const int k = step[w];
    if (k >= steps) return false;
    if (!sent[w]) {
      for (int j = w; j < m; j += nw)
        if (bd::coop_exchanged(m, nw, k, j)) slot[k & 1][j] = k + 1;
      sent[w] = 1;
      return true;
    }
    for (int j = 0; j < m; ++j)
      if (bd::coop_exchanged(m, nw, k, j) && slot[k & 1][j] != k + 1) return false;
    step[w] = k + 1;
    sent[w] = 0;
    return true;
  };
  for (;;) {
    bool moved = false;
    for (int w = 0; w < nw; ++w)
      if (w != late) moved |= advance(w);
    if (!moved && !advance(late)) break;
  }
  for (int w = 0; w < nw; ++w)
    if (step[w] < steps) return false;
  return true;
}
int main() {
  for (int m = 3; m <= 70; ++m)
    for (int nw = 1; nw <= (m < 32 ? m : 32); ++nw) {
      for (int k = 0; k < m - 2; ++k)
        for (int j = k + 1; j < m; ++j)
          if (!bd::coop_exchanged(m, nw, k, j)) return std::printf("m=%d nw=%d k=%d: y_%d not exchanged\n", m, nw, k, j), 1;
      for (int late = 0; late < nw; ++late)
        if (!finishes(m, nw, late)) return std::printf("m=%d nw=%d: worker %d left behind\n", m, nw, late), 1;
    }
  return 0;
}
"""


def test_no_worker_is_left_behind(tmp_path):
    source, program = tmp_path / "exchange.cpp", tmp_path / "exchange"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(source), "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout
