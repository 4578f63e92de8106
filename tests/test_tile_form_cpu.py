"""How the weights-in-registers kernel would run a launch, at the borders where its epilogues change."""
from host_program import run_host

PROGRAM = r"""
#include "kernels.h"
#include <cstdio>
using namespace ohip;
alignas(16) static char any[16];
static void show(DType in, DType out, int rows, int k, int columns, bool residual) {
  IgemmParams p;   // a product of rows x k x columns
  p.in_dt = in; p.out_dt = out;
  p.N = rows; p.H = p.W = p.Ho = p.Wo = 1;
  p.C = p.xcs = k;
  p.R = p.S = p.sh = p.sw = p.dh = p.dw = 1;
  p.Kout = p.ycs = p.rcs = columns;
  p.w_rows = columns; p.w_cols = p.w_rs = k;
  p.wf_chunks = k * dtype_size(in) / 32; p.wf_tiles = (columns + 31) / 32;
  p.batch = 1;
  if (residual) p.residual = any;
  const WregForm f = igemm_wreg_form(p);
  printf("%d %d %d %d | %d %d\n", dtype_size(out), rows, columns, (int)residual, f.rows, f.epilogue);
}
int main() {
  for (DType out : {DT_BF16, DT_F32}) {
    // 256 workgroups, one per compute unit, and the next number of them
    show(DT_BF16, out, 4096, 256, 1024, true);
    show(DT_BF16, out, 4097, 256, 1024, true);
    show(DT_BF16, out, 8192, 256, 1024, true);
    // without a residual: two per compute unit, and more
    show(DT_BF16, out, 8192, 256, 1024, false);
    show(DT_BF16, out, 10240, 256, 1024, false);
  }
}
"""


def test_epilogue_follows_the_workgroups(tmp_path):
    got = [tuple(int(v) for v in line.split("|")[1].split()) for line in run_host(tmp_path, PROGRAM).splitlines()]
    epilogue = [g[1] for g in got]
    # 2 = residual ahead of the K loop, 1 = accumulator layout, 0 = by rows
    assert epilogue[:5] == [2, 0, 0, 1, 1], got
    assert epilogue[5:] == [2, 0, 0, 1, 0], got
