"""Small C++ programs against the host side of the kernels' interface (csrc/kernels/kernels.h),
linked with the built library: what a launcher or a dispatch rule decides, without a launch."""
import os
import subprocess

import __graft_entry__ as entry


def run_host(tmp_path, source):
    """Compile, run, return what it printed."""
    entry.load().odla.load_library()
    src, exe = tmp_path / "host.cc", tmp_path / "host"
    src.write_text(source)
    lib, kernels = entry.PKG_DIR, os.path.join(entry.PKG_DIR, "csrc", "kernels")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + kernels, str(src), "-L" + lib, "-lodla_hip",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib, "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)], check=True, timeout=120)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout
