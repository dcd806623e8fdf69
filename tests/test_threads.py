"""Host threads of one call: when a thread cannot be started because memory has run
out, the ones there are do the work and nothing ends the process."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcf_amd", "csrc")

PROGRAM = r"""
#include "sdpd_threads.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
static std::atomic<int> left{1 << 30};
void* operator new(std::size_t n) {
  if (left.fetch_sub(1) <= 0) throw std::bad_alloc();
  return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main(int, char** argv) {
  left = std::atoi(argv[1]);
  std::atomic<int> next{0}, done{0};
  auto work = [&](int) {
    while (next.fetch_add(1) < 100) done.fetch_add(1);
  };
  sdpd::run_slots<8>(std::atoi(argv[2]), work);
  left = 1 << 30;
  std::printf("%d\n", done.load());
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("threads")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-o", str(d / "t"), str(d / "t.cpp"),
                    "-lpthread"], check=True)
    return str(d / "t")


@pytest.mark.parametrize("allocations", [0, 1, 3, 1000])
@pytest.mark.parametrize("slots", [1, 2, 8])
def test_every_piece_is_done(program, allocations, slots):
    r = subprocess.run([program, str(allocations), str(slots)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stderr
    assert r.stdout == "100\n"
