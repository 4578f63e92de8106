"""The row kernel of a product without an activation holds none of their code: such a launch is one
call of a few microseconds, and what it would jump over is fetched from memory on its way."""
import os
import re
import subprocess

import pytest

import __graft_entry__ as entry
from test_igemm_codegen import FLAGS, HIPCC


def test_products_without_an_activation_are_short(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    src, out = os.path.join(entry.PKG_DIR, "csrc", "kernels", "gemm_rowdot.hip"), str(tmp_path / "rowdot.s")
    subprocess.run([HIPCC] + FLAGS + [src, "-o", out], check=True, capture_output=True, timeout=300)
    size = {}
    for body in re.split(r"; -- Begin function ", open(out).read())[1:]:
        name, length = body.split("\n")[0], re.search(r"codeLenInByte = (\d+)", body)
        kernel = re.search(r"gemm_rowdot_kernelILi(\d+)ELb([01])E", name)
        if kernel and length:
            size[int(kernel.group(1)), kernel.group(2) == "1"] = int(length.group(1))
    assert sorted(size) == [(4, False), (4, True), (8, False), (8, True), (16, False), (16, True)]
    for (columns, act), n in size.items():
        assert act or n <= 1024 + 256 * columns, size   # (sums: up to 200 bytes per column)
