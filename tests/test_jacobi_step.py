"""The rotation of the canonicalisers' Jacobi (csrc/jacobi.hpp), compiled for the CPU with the hardware's reciprocal
estimates played by exact ones that are off by their documented 2^-22: tangent, cosine, sine and phase to rounding."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

STUB = r"""
#pragma once
#include <cmath>
#include <cstdlib>
#define __device__
#define __forceinline__ inline
using std::fma;
inline double off(double y) { return y * (1.0 + std::ldexp(2.0 * std::rand() / RAND_MAX - 1.0, -22)); }
inline double estimate_rsq(double x) { return off(1.0 / std::sqrt(x)); }
inline double estimate_rcp(double x) { return off(1.0 / x); }
#define __builtin_amdgcn_rsq estimate_rsq
#define __builtin_amdgcn_rcp estimate_rcp
"""

PROGRAM = r"""
#include "jacobi.hpp"
#include <cstdio>
typedef long double L;

int main() {
  const L u = 1.1102230246251565e-16L;   // unit of rounding
  L worst_t = 0, worst_c = 0, worst_s = 0, worst_e = 0, worst_g = 0;
  for (int k = 0; k < 400000; ++k) {
    auto uni = [] { return (double)std::rand() / RAND_MAX; };
    // squared norms over 26 decades, cosines from the settled threshold and below to one
    const double a = std::pow(10.0, -26 * uni()), b = k % 5 ? std::pow(10.0, -26 * uni()) : a * (1 + 1e-9 * uni());
    const double cosine = std::pow(10.0, -14 * uni()), phase = 6.283185307179586 * uni(), g = cosine * std::sqrt(a) * std::sqrt(b);
    const double gr = g * std::cos(phase), gi = g * std::sin(phase), g2 = gr * gr + gi * gi;
    const bqa::JacobiStep j = bqa::jacobi_step(a, b, gr, gi, g2);
    const L ga = std::sqrt((L)g2), zeta = ((L)b - (L)a) / (2 * ga);
    const L t = (zeta < 0 ? -1 : 1) / (std::fabs(zeta) + std::sqrt(zeta * zeta + 1)), c = 1 / std::sqrt(t * t + 1);
    auto rel = [&](L x, L y) { return std::fabs(x / y - 1); };
    worst_t = std::fmax(worst_t, rel(j.t, t));
    worst_c = std::fmax(worst_c, rel(j.c, c));
    worst_s = std::fmax(worst_s, rel(j.s, c * t));
    worst_g = std::fmax(worst_g, rel(j.tg, t * ga));
    worst_e = std::fmax(worst_e, std::fmax(std::fabs(j.er - gr / ga), std::fabs(j.ei + gi / ga)));
  }
  std::printf("units of rounding: t %.2Lf c %.2Lf s %.2Lf t|g| %.2Lf e %.2Lf\n", worst_t / u, worst_c / u, worst_s / u,
              worst_g / u, worst_e / u);
  // a reciprocal (root) is good to two units.  t: the root, the product and the difference of zeta (b - a is rounded
  // once), h with its root and product, their sum, the reciprocal, where h counts half: ten units; c two more at half of
  // t's, s and t|g| a product or two more
  return worst_t < 10 * u && worst_c < 8 * u && worst_s < 16 * u && worst_g < 16 * u && worst_e < 4 * u ? 0 : 1;
}
"""


def test_step_is_exact_to_rounding(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(STUB)
    src, exe = tmp_path / "step.cpp", tmp_path / "step"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-ffp-contract=off", "-I", str(tmp_path), "-I",
                    os.path.join(ROOT, "bqa_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    print(done.stdout)
    assert done.returncode == 0, done.stdout
