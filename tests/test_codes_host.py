"""CPU checks of the 16-bit codes' arithmetic (compiled for the host from the
kernels' header): the bitmap byte of any 16 bits lies inside the bitmap, every
vertex has a bit of its own, and the lists of codes stay inside their pool up
to its largest size."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "tc_kernels.hpp"
using namespace tck;

static int bad(const char* what, long long a, long long b) {
  std::printf("%s: %lld %lld\n", what, a, b);
  return 1;
}

int main() {
  for (long long n : {1LL, 2LL, 8191LL, 8192LL, 8193LL, 16384LL, 16385LL, 32768LL, 32769LL, 65534LL, 65535LL}) {
    const int kb = core_bits(n);
    if (((long long)8 << kb) < n) return bad("bitmap too small", n, kb);
    // what a load may hold besides codes: any word
    for (uint32_t w = 0; w < 65536; ++w)
      if (code_byte(w | 0xFFFF0000u, 0, kb) >= 1u << kb || code_byte(w << 16 | 0xFFFFu, 1, kb) >= 1u << kb)
        return bad("byte past the bitmap", w, kb);
    std::vector<bool> seen((size_t)8 << kb);
    for (long long i = 0; i < n; ++i) {
      const uint32_t c = core_code((uint32_t)i, kb);
      if (c > 65535u || c == kNoCode || code_byte(c, 0, kb) != (c & 0x1FFFu) || code_byte(c << 16, 1, kb) != (c & 0x1FFFu))
        return bad("code of vertex", i, c);
      const size_t bit = 8 * (size_t)(c & 0x1FFFu) + (c >> kCoreByteBits);
      if (seen[bit]) return bad("two vertices on one bit", i, c);
      seen[bit] = true;
    }
  }
  // lists of n codes, one after another: each inside [2p, 2p + 2n), at the
  // pool's beginning and where its positions are largest
  for (long long p0 : {0LL, 1LL, 12345LL, (long long)kCorePool - 70000}) {
    long long p = p0;
    for (uint32_t n = 0; n < 360 && p + n < kCorePool; p += n, n += n < 200 ? 1 : 37) {
      const uint32_t s = code_start(p, n);
      if ((long long)s < 2 * p || (n && (long long)s + n > 2 * p + 2 * (long long)n)) return bad("list of codes", p, n);
      if ((uint64_t)s * 2 + 2 * n >= (uint64_t)1 << 32) return bad("byte offset of a list", p, n);
      const int64_t l = line_start(p, (int32_t)n);
      if (l < 2 * p || (n && l + n > 2 * p + 2 * (long long)n)) return bad("list on lines", p, n);
      if (n && n <= 32 && l / 32 != (l + n - 1) / 32) return bad("list over two lines", p, n);
    }
  }
  return 0;
}
"""


def test_code_arithmetic(tmp_path):
    src, exe = tmp_path / "codes.cpp", tmp_path / "codes"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "hetegeneous_parallel_programming_amd", "csrc", "hip"),
                    str(src), "-o", str(exe)], check=True, capture_output=True, text=True, timeout=300)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout
