"""The rule of a job's kept graphs (csrc/graph_cache.hpp), compiled for the CPU: what a run holds outlives its own
additions, and every graph is destroyed once."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include "graph_cache.hpp"
#include <cstdio>
#include <set>

std::set<int> alive;
int made = 0;
bool ok = true;
void destroy(int g) { ok = ok && alive.erase(g) == 1; }

template <size_t CAP>
int take(bqa::GraphCache<int, CAP>& c, intptr_t bond, intptr_t sweeps) {
  if (int* g = c.find({bond, sweeps})) return *g;
  alive.insert(++made);
  c.add({bond, sweeps}, made, destroy);
  return made;
}

template <size_t CAP>
void runs() {
  {
    bqa::GraphCache<int, CAP> c;
    // every order of ten bond dimensions that a small generator gives: a run takes its short graph, then its long one
    unsigned x = 1;
    for (int k = 0; k < 2000; ++k) {
      x = x * 1103515245u + 12345u;
      const int bond = (x >> 16) % 10;
      const bool lengthy = (x >> 8) % 3 != 0;
      const int a = take(c, bond, 4);
      const int b = lengthy ? take(c, bond, 16) : a;
      ok = ok && alive.count(a) == 1 && alive.count(b) == 1 && alive.size() <= CAP;
      if (int* again = c.find({bond, 4})) ok = ok && *again == a;
      else ok = false;
    }
    c.clear(destroy);
  }
  ok = ok && alive.empty();
}

int main() {
  runs<2>();
  runs<3>();
  runs<8>();
  std::puts(ok ? "ok" : "bad");
  return ok ? 0 : 1;
}
"""


def test_a_run_keeps_its_graphs(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "cache.cpp", tmp_path / "cache"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "bqa_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True).stdout.strip() == "ok"
