"""Which compiled window a pool of a plane chain runs with: the one of its own size and step, or the
loop that takes both from the arguments."""
from host_program import run_host

PROGRAM = r"""
#include "kernels.h"
#include <cstdio>
using namespace ohip;
int main() {
  for (int is_max = 0; is_max < 2; ++is_max)
    for (int kh = 1; kh <= 5; ++kh)
      for (int kw = 1; kw <= 5; ++kw)
        for (int sh : {1, 2, 3, 10, 11, 12, 21, 22, 31, 32})
          for (int sw : {1, 2, 3, 10, 11, 12, 21, 22, 31, 32})
            for (int pad = 0; pad < 2; ++pad) {
              PlaneGroup g;
              g.chunks = g.n_inst = 1;
              PlaneInst& I = g.inst[0];
              I.kind = PLANE_POOL;
              I.is_max = is_max;
              I.H = I.W = 100;
              I.kh = kh; I.kw = kw; I.sh = sh; I.sw = sw; I.ph = I.pw = pad;
              I.Ho = (I.H + 2 * pad - kh) / sh + 1;
              I.Wo = (I.W + 2 * pad - kw) / sw + 1;
              plane_prepare(&g);
              printf("%d %d %d %d %d %d %d %d\n", is_max, kh, kw, sh, sw, pad, I.Wo, I.window);
            }
}
"""

# window number -> size, step, maximum, whether it takes no taps outside the plane
COMPILED = {1: (1, 1, 0, True), 2: (2, 1, 0, True), 3: (2, 2, 0, True), 4: (3, 2, 0, False), 5: (2, 2, 1, False), 6: (3, 2, 1, False), 7: (3, 1, 1, False)}


def test_compiled_windows_have_the_size_and_step_of_the_pool(tmp_path):
    seen = set()
    for line in run_host(tmp_path, PROGRAM).splitlines():
        is_max, kh, kw, sh, sw, pad, wo, window = map(int, line.split())
        if window not in COMPILED:
            assert window == (8 if is_max else 9), line
            continue
        size, step, maximum, inside = COMPILED[window]
        assert (kh, kw, sh, sw, is_max) == (size, size, step, step, maximum) and wo >= 4 and not (inside and pad), line
        seen.add(window)
    assert seen == set(COMPILED)
