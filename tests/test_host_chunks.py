"""How transfers of raw arrays are cut into chunks (csrc/host_chunks.h), on the
CPU: the chunks cover every site once and stay inside a pinned buffer and the
staging, also those of some of the arrays in the staging of all of them (the long
links read a second time when they turn out not to be SU(3))."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "milc-qphix_amd", "csrc")
PROGRAM = r"""
#include "host_chunks.h"
#include <cstdio>
using namespace qphix;
static long bad = 0, cases = 0;
static void check(size_t per, size_t half, int halves, size_t stage) {
  const HostPlan p = host_plan(per, half, halves);
  size_t at = 0;
  for (size_t c = 0; c < p.chunks; ++c) {
    const size_t first = p.first(c), n = p.count(c), b = c % p.nbuf;
    const bool ok = first == at && n > 0 && first / half == (first + n - 1) / half &&
                    p.chunk * per <= HOST_CHUNK && per * p.chunk * b + per * n <= stage &&
                    (n % 64 == 0 || half % 64 != 0);
    if (!ok && !bad++) std::printf("per %zu half %zu x %d: chunk %zu of %zu\n", per, half, halves, c, p.chunks);
    at = first + n;
  }
  if (at != half * halves && !bad++) std::printf("per %zu half %zu x %d: %zu sites\n", per, half, halves, at);
  ++cases;
}
int main() {
  const size_t one[] = {24, 48, 288, 576};  // FP32 and FP64 vectors, links
  for (size_t half = 128; half < 6000000; half = (half * 9 / 8 + 127) / 128 * 128)
    for (int halves = 1; halves <= 2; ++halves)
      for (size_t s : one)
        for (size_t n = 1; n <= 4; ++n) {
          const size_t stage = host_stage_bytes(n * s, half, halves);
          for (size_t m = 1; m <= n; ++m) check(m * s, half, halves, stage);
        }
  std::printf("%ld cases, %ld bad\n", cases, bad);
  return bad != 0;
}
"""


def test_chunks_stay_inside_their_buffers(tmp_path):
    src, exe = tmp_path / "chunks.cpp", tmp_path / "chunks"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", exe, src], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
