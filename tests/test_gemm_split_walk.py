"""What the waves of gemm_split.hip read of B (gemm_split_walk.hpp), walked on the CPU: with a range check that sees the vector offset
only, no dword that passes it lies outside the matrix, and every element that a product needs is read from its place."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncv_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <initializer_list>
#include "gemm_split_walk.hpp"
using namespace nncv_hip;
int main() {
  for (int K : {1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 65, 97, 353, 369})
    for (int N : {1, 2, 31, 63, 64, 65, 190})
      for (int TN : {1, 2})
        for (int KG : {1, 4, 8})
          for (int n0 = 0; n0 < N; n0 += 32 * TN)
            for (int grp = 0; grp < KG; ++grp) {
              bool last = true;
              for (int r = (K + 31) / 32 - 1 - grp;; r -= KG) {  // as a wave walks them, one round past its first included
                for (int k = 0; k < 2; ++k) {
                  const SplitBRows b = split_b_rows(r, k, n0, N, K);
                  for (int lane = 0; lane < 64; ++lane)
                    for (int e = 0; e < 8; ++e)
                      for (int j = 0; j < TN; ++j) {
                        const unsigned v = split_b_vector(split_b_lane(lane, TN, n0, N), e, N, last) + 4u * j, s = split_b_scalar(e, N, last);
                        const bool read = (unsigned long long)v + 4 <= b.bytes;
                        const long long at = b.first * 4 + v + s, row = 32ll * r + 16 * k + 8 * (lane / 32) + e, col = n0 + TN * (lane % 32) + j;
                        if (read && (at < 0 || at + 4 > 4ll * K * N)) return printf("K %d N %d TN %d KG %d round %d: byte %lld of %lld\n", K, N, TN, KG, r, at, 4ll * K * N), 1;
                        if (row >= 0 && row < K && col < N && (!read || at != (row * N + col) * 4)) return printf("K %d N %d TN %d: element %lld %lld\n", K, N, TN, row, col), 1;
                      }
                }
                if (r < 0) break;
                last = false;
              }
            }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_no_read_leaves_the_matrix(tmp_path):
    (tmp_path / "driver.cpp").write_text(DRIVER)
    exe = str(tmp_path / "driver")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(tmp_path / "driver.cpp"), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
