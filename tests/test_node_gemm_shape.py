"""Which classes the matrix-product kernels serve (csrc/node_gemm_shape.hpp), compiled for the CPU: their workspace is
small, or no larger than the generic kernels', and small tensors of many nodes are left to those."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = r"""
#include "node_gemm_shape.hpp"
#include <cstdio>
#include <initializer_list>
using namespace bqa;

int main() {
  int served = 0, refused = 0;
  for (int d = 1; d <= 7; ++d)
    for (int chi = 1; chi <= 40; ++chi)
      for (int n : {1, 2, 3, 4, 5, 8, 100, 1024, 5000}) {
        if (!gemm_fits(n, d, chi)) {
          refused += gemm_shape(d, chi);
          continue;
        }
        ++served;
        double tensor = 2;
        for (int k = 0; k < d; ++k) tensor *= chi;
        const double generic = 3.0 * (n < 1024 ? n : 1024) * tensor * 16;
        for (size_t element : {8, 16}) {
          const int chunk = gemm_chunk(n, d, chi, element);
          const double bytes = (double)chunk * gemm_node_bytes(d, chi, element);
          if (chunk < 1 || chunk > n || gemm_node_bytes(d, chi, element) != element * gemm_products(d) * tensor ||
              bytes > (generic > 4.0 * (1u << 30) ? generic : 4.0 * (1u << 30))) {
            std::printf("d %d chi %d n %d: chunk %d, %g bytes, generic %g\n", d, chi, n, chunk, bytes, generic);
            return 1;
          }
        }
      }
  // a single hub of degree 6 at chi = 24 (6 GB in FP64, 73 GB of products) and the shapes of ordinary graphs
  if (gemm_fits(1, 6, 24) || gemm_fits(2, 6, 24) || !gemm_fits(4, 6, 24) || !gemm_fits(1, 5, 24) || !gemm_fits(1, 4, 32) ||
      !gemm_fits(120, 5, 8) || !gemm_fits(100, 3, 32))
    return 2;
  // tensors above 2,048 elements never go back to the generic kernel for being small, nor any below for few nodes in BP
  for (GemmUse use : {kGemmBp, kGemmExt, kGemmDensity})
    for (int d = 2; d <= 6; ++d)
      for (int chi = 2; chi <= 32; ++chi) {
        double tensor = 2;
        for (int k = 0; k < d; ++k) tensor *= chi;
        for (int n : {1, 100, 300, 1024, 100000})
          for (size_t element : {8, 16})
            if (gemm_too_small(use, n, d, chi, element) && (tensor > 2048 || (use != kGemmDensity && (n <= 100 || tensor > 512))))
              return 4;
      }
  // FP32 products are summed with more bits than the generic kernel's
  for (GemmUse use : {kGemmBp, kGemmDensity})
    if (gemm_too_small(use, 5000, 2, 9, 8) || gemm_too_small(use, 5000, 6, 2, 8)) return 6;
  if (!gemm_too_small(kGemmBp, 578, 5, 2, 16) || gemm_too_small(kGemmBp, 120, 5, 2, 16) || gemm_too_small(kGemmBp, 3000, 5, 4, 16) ||
      !gemm_too_small(kGemmBp, 1200, 2, 13, 16) || gemm_too_small(kGemmBp, 1200, 2, 13, 8) || gemm_too_small(kGemmBp, 10000, 2, 13, 16) ||
      !gemm_too_small(kGemmExt, 3000, 5, 3, 16) || gemm_too_small(kGemmExt, 600, 5, 3, 16) || gemm_too_small(kGemmExt, 3000, 3, 9, 16) ||
      !gemm_too_small(kGemmDensity, 20, 5, 2, 16) || gemm_too_small(kGemmDensity, 20, 5, 4, 16) || gemm_too_small(kGemmDensity, 3000, 3, 9, 8))
    return 5;
  std::printf("%d %d\n", served, refused);
  return served > 0 && refused > 0 ? 0 : 3;
}
"""


def test_workspace_stays_within_the_generic_kernels(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "shape.cpp", tmp_path / "shape"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Wextra", "-Werror", "-Wno-unused-function", "-I",
                    os.path.join(ROOT, "bqa_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
