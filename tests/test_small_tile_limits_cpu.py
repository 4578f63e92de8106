"""Where the small tiles are declined because their 32-bit buffer offsets would not reach: the images a
tile of 32 pixels can touch span 2^31 bytes, or a row of weights 2^25."""
from host_program import run_host

PROGRAM = r"""
#include "kernels.h"
#include <cstdio>
using namespace ohip;
static int variant(DType dt, int n, int h, int w, int c) {
  IgemmParams p;   // 1x1 filters whose step leaves one pixel of an image
  p.in_dt = p.out_dt = dt;
  p.N = n; p.H = h; p.W = w; p.C = p.xcs = c;
  p.Ho = p.Wo = 1; p.sh = h; p.sw = w;
  p.R = p.S = p.dh = p.dw = 1;
  p.Kout = p.ycs = 64;
  p.w_rows = 64; p.w_cols = c; p.w_rs = c;
  p.batch = 1;
  return igemm_slim_variant(p, true);
}
int main() {
  const int e = 64;
  for (DType dt : {DT_F16, DT_BF16, DT_F32, DT_I8}) {
    const int s = dtype_size(dt), side = 8 / s;   // 2^31 bytes are side * 2^22 pixels of 64 channels
    printf("image %d %d %d\n", s, variant(dt, 1, side << 10, 4095, e) > 0, variant(dt, 1, side << 10, 4096, e) > 0);
    printf("images4 %d %d %d\n", s, variant(dt, 4, side << 9, 2047, e) > 0, variant(dt, 4, side << 9, 2048, e) > 0);
    printf("images32 %d %d %d\n", s, variant(dt, 32, side << 8, 511, e) > 0, variant(dt, 32, side << 8, 512, e) > 0);
    printf("images100 %d %d %d\n", s, variant(dt, 100, side << 8, 511, e) > 0, variant(dt, 100, side << 8, 512, e) > 0);
    printf("weights %d %d %d\n", s, variant(dt, 1, 1, 1, (1 << 25) / s - 16) > 0, variant(dt, 1, 1, 1, (1 << 25) / s) > 0);
  }
}
"""


def test_taken_below_the_limit_and_declined_at_it(tmp_path):
    lines = run_host(tmp_path, PROGRAM).splitlines()
    assert len(lines) == 20
    for line in lines:
        assert line.split()[2:] == ["1", "0"], line
