"""The quotients by multiplication of csrc/gsg_index.hpp against C's division (host).

Every divisor k^d and every dividend below k^D of the transforms (k in {2, 3, 5}, D <= 8),
and the dividends next to the multiples of each divisor, largest first, below 2^31."""
import subprocess

from conftest import ROOT

CODE = r"""
#include "gsg_index.hpp"
#include <cstdio>
#include <initializer_list>
using namespace gsg;
int main() {
  long bad = 0;
  for (uint32_t k : {2u, 3u, 5u}) {
    uint32_t top = 1;
    for (int D = 1; D <= 8; ++D) top *= k;
    for (uint32_t d = k; d <= top; d *= k) {
      const QuotMul q = quot_mul(d);
      for (uint32_t n = 0; n < top; ++n) bad += quot(n, q) != n / d;
      for (uint32_t m = (1u << 31) / d, i = 0; m > 0 && i < 200000; --m, ++i)
        for (uint32_t n : {m * d - 1, m * d, m * d + 1}) bad += n < (1u << 31) && quot(n, q) != n / d;
    }
  }
  std::printf("%ld\n", bad);
  return bad != 0;
}
"""


def test_quotients_are_exact(tmp_path):
    src, exe = tmp_path / "q.cpp", tmp_path / "q"
    src.write_text(CODE)
    inc = ROOT / "galerkinsparsegrids.jl_amd" / "csrc"
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{inc}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
