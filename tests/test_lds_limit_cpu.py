"""A kernel's LDS limit is raised once on every device it is launched on, whichever thread comes
first: kernels/lds_limit.h against stand-ins of the two runtime calls it makes."""
import os
import subprocess

import __graft_entry__ as entry

PROGRAM = r"""
#include "lds_limit.h"
#include <cstdio>
#include <thread>
#include <vector>
static thread_local int t_device = 0;
static std::atomic<int> raised[70], fails{0};
extern "C" hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
  if (fails.load() > 0) { --fails; return hipErrorInvalidValue; }
  ++raised[t_device];
  return hipSuccess;
}
int main() {
  static ohip::LdsLimit limit;
  fails = 1;
  if (limit.raise(&limit, 1) == hipSuccess) return 1;   // an error is reported, and not kept as done
  for (int round = 0; round < 3; ++round)
    for (int d : {0, 1, 7, 63}) {
      t_device = d;
      if (limit.raise(&limit, 1) != hipSuccess) return 2;
      if (raised[d] != 1) return 3;
    }
  t_device = 69;
  for (int i = 1; i < 4; ++i)
    if (limit.raise(&limit, 1) != hipSuccess || raised[69] != i) return 4;
  static ohip::LdsLimit shared;
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&, t] {
      t_device = 10 + t % 2;
      for (int i = 0; i < 1000; ++i)
        if (shared.raise(&shared, 1) != hipSuccess || raised[t_device] < 1) ++bad;
    });
  for (auto& t : ts) t.join();
  return bad.load() == 0 ? 0 : 5;
}
"""


def test_limit_is_raised_once_per_device(tmp_path):
    src, exe = tmp_path / "limit.cc", tmp_path / "limit"
    src.write_text(PROGRAM)
    kernels = os.path.join(entry.PKG_DIR, "csrc", "kernels")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + kernels,
                    str(src), "-o", str(exe)], check=True, timeout=120)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0


def test_no_launch_keeps_such_a_flag_of_its_own():
    kernels = os.path.join(entry.PKG_DIR, "csrc", "kernels")
    for f in sorted(os.listdir(kernels)):
        if f != "lds_limit.h":
            assert "hipFuncSetAttribute" not in open(os.path.join(kernels, f)).read(), f
