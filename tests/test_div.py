"""The division by a fixed divisor that finds a tile's coordinates (Div and
div_by in csrc/common.hpp), compiled for the host: against integer division at
the divisors and numerators where the multiplier could be one too small."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = """
#include <cstdint>
#include <cstdio>
#define __host__
#define __device__
%s
int main() {
  const int64_t LIM = (int64_t)1 << 31;
  long long bad = 0;
  auto check = [&](int64_t d) {
    const Div q(d);
    auto one = [&](int64_t n) { if (n >= 0 && n < LIM && div_by((uint32_t)n, q) != (uint32_t)(n / d)) bad++; };
    for (int64_t k = 0; k < 4; k++) {
      one(k); one(LIM - 1 - k); one(d - 2 + k); one(LIM / 2 - 2 + k);
    }
    for (int64_t i = 1, m = LIM / d; i < 64; i++)  // around multiples of d over the whole range
      for (int64_t k = -1; k < 2; k++) { one(m * i / 64 * d + k); one(m * d + k); }
  };
  for (int64_t d = 1; d < 70000; d++) check(d);
  for (int s = 1; s < 32; s++)
    for (int64_t k = -3; k < 4; k++) if (((int64_t)1 << s) + k > 0) check(((int64_t)1 << s) + k);
  uint64_t r = 1;
  for (int i = 0; i < 200000; i++) {
    r = r * 6364136223846793005ull + 1442695040888963407ull;
    check(1 + (int64_t)(r >> 33) %% (LIM - 1));
  }
  printf("%%lld\\n", bad);
  return bad != 0;
}
"""


def test_division(tmp_path):
  text = open(os.path.join(ROOT, "connected-components-3d_amd", "csrc", "common.hpp")).read()
  div = re.search(r"struct Div \{.*?\n\};\n__device__ inline uint32_t div_by\(.*?\n", text, flags=re.S).group(0)
  src = tmp_path / "div.cpp"
  src.write_text(MAIN % div)
  exe = tmp_path / "div"
  subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(src)], check=True)
  assert subprocess.run([str(exe)], capture_output=True, text=True).stdout.strip() == "0"
