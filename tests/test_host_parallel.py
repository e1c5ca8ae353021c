"""The host threads of the triangular solves' planning: a process that can start
no more threads, and one out of memory inside a thread, get the loop done and an
exception of the caller's, not an abort."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "psblas3_amd",
                    "csrc")
DRIVER = r"""
#include <stdio.h>
#include <string.h>
#include <sys/resource.h>
#include <atomic>
#include <new>
#include "host_parallel.hpp"
int main(int argc, char** argv) {
  if (!strcmp(argv[1], "no_threads")) {     // room for no thread's stack
    long pages = 0;
    FILE* f = fopen("/proc/self/statm", "r");
    if (!f || fscanf(f, "%ld", &pages) != 1) return 2;
    fclose(f);
    rlimit lim;
    lim.rlim_cur = lim.rlim_max = (rlim_t)pages * 4096 + (2 << 20);
    if (setrlimit(RLIMIT_AS, &lim)) return 2;
  }
  const int n = 100003;
  std::atomic<long> sum{0}, ranges{0};
  try {
    psbhip::host_parallel(n, 10, [&](int k, int lo, int hi) {
      if (!strcmp(argv[1], "throws") && lo <= n - 1 && n - 1 < hi) throw std::bad_alloc();
      long s = 0;
      for (int i = lo; i < hi; i++) s += i;
      sum += s;
      ranges++;
    });
  } catch (const std::bad_alloc&) {
    puts("bad_alloc");
    return 0;
  }
  printf("%ld %d\n", sum.load(), ranges.load() > 1);
  return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_parallel")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I" + CSRC,
                           str(d / "driver.cpp"), "-o", str(d / "driver")])
    return str(d / "driver")


@pytest.mark.parametrize("mode", ["usual", "no_threads"])
def test_every_range_runs(driver, mode):
    out = subprocess.run([driver, mode], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    assert out.stdout.split()[0] == str(100003 * 100002 // 2)


def test_exception_reaches_the_caller(driver):
    out = subprocess.run([driver, "throws"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "bad_alloc\n", out.stderr
