"""The host threads of the raw transfers (csrc/copy_pool.h), on the CPU: copies of
all sizes are complete on return, with every number of threads; a process that
gets no more threads goes on with those it has; and a pool can be destroyed while a
transfer is open."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "milc-qphix_amd", "csrc")
PROGRAM = r"""
#include "copy_pool.h"
#include <cstdio>
#include <cstdlib>
#include <sys/resource.h>
using namespace qphix;
static const size_t most = 9 * HOST_SLICE + 77;
static char s[most], d[most];
static int copies(CopyPool &pool) {
  for (size_t k = 0; k < most; ++k) s[k] = (char)(k * 2654435761u >> 13);
  const size_t sizes[] = {0, 1, 4095, HOST_SLICE - 1, HOST_SLICE, HOST_SLICE + 1, 3 * HOST_SLICE + 5, most};
  for (int round = 0; round < 50; ++round) {
    pool.open();
    for (size_t n : sizes) {
      std::memset(d, round, most);
      pool.copy(d, s, n);
      if (std::memcmp(d, s, n) != 0) return 1;
      for (size_t k = n; k < most; ++k)
        if (d[k] != (char)round) return 1;
    }
    pool.close();
  }
  return 0;
}
int main(int argc, char **argv) {
  const int workers = std::atoi(argv[1]);
  if (argc > 2) {  // room for a few thread stacks
    rlimit r{(rlim_t)96 << 20, (rlim_t)96 << 20};
    if (setrlimit(RLIMIT_AS, &r) != 0) return 2;
  }
  CopyPool pool(workers);
  if (int rc = copies(pool)) return rc;
  pool.open();  // destroyed during a transfer: its threads end all the same
  pool.copy(d, s, most);
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "pool.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", CSRC, "-o", d / "pool", d / "pool.cpp"],
                   check=True)
    return str(d / "pool")


@pytest.mark.parametrize("workers", [0, 1, 7])
def test_copies(program, workers):
    assert subprocess.run([program, str(workers)], timeout=60).returncode == 0


def test_no_more_threads(program):
    assert subprocess.run([program, "64", "limited"], timeout=60).returncode == 0
