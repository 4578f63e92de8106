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


PAIR_PROGRAM = r"""
#include "kernels.h"
#include <cstdio>
#include <map>
// stand-ins of the runtime's calls behind a launch
static std::map<const void*, size_t> limit;
static size_t pushed = 0, launches = 0, beyond = 0;
extern "C" hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int bytes) { limit[f] = (size_t)bytes; return hipSuccess; }
extern "C" hipError_t __hipPushCallConfiguration(dim3, dim3, size_t lds, hipStream_t) { pushed = lds; return hipSuccess; }
extern "C" hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  *g = *b = dim3(1); *lds = pushed; *s = nullptr;
  return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {
  ++launches;
  if (lds > 65536 && limit[f] < lds) { std::fprintf(stderr, "%zu bytes, limit %zu\n", lds, limit[f]); ++beyond; }
  if (limit[f] > 160 * 1024) ++beyond;
  return hipSuccess;
}
int main() {
  using namespace ohip;
  void* at = reinterpret_cast<void*>(0x100000);   // (never read)
  for (DType dt : {DT_F16, DT_BF16})
    for (int wide : {128, 256})
      for (int narrow : {64, 128})
        for (int form : {0, 1, 2}) {
          if (form == 2 && narrow == 128) continue;
          IgemmParams p;
          p.in_dt = p.out_dt = dt;
          p.N = 1; p.H = p.W = p.Ho = p.Wo = 5;
          p.C = p.xcs = 64; p.Kout = p.ycs = p.rcs = wide; p.wf_chunks = 4;
          p.f_kout = p.f_ycs = narrow; p.f_wf_chunks = wide / 16;
          p.x = p.y = p.f_y = at; p.w_frag = p.f_wfrag = at;
          if (form == 1) p.residual = at;
          if (form == 2) { p.r_x = at; p.r_wfrag = at; p.r_xcs = 64; }
          if (launch_igemm_pair(p, nullptr) != hipSuccess) return 1;
        }
  return launches == 20 && beyond == 0 ? 0 : 2;
}
"""


def test_pair_of_pointwise_layers_raises_its_limit(tmp_path):
    """Every instance of the kernel may use the LDS that its launch asks for."""
    src, exe = tmp_path / "pair.cc", tmp_path / "pair"
    src.write_text(PAIR_PROGRAM)
    entry.load().odla.load_library()
    lib = os.path.join(entry.PKG_DIR, "libodla_hip.so")
    kernels = os.path.join(entry.PKG_DIR, "csrc", "kernels")
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + kernels, str(src), lib,
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,%s:/opt/rocm/lib" % entry.PKG_DIR, "-o", str(exe)], check=True, timeout=120)
    done = subprocess.run([str(exe)], timeout=60, stderr=subprocess.PIPE, text=True)
    assert done.returncode == 0, done.stderr
