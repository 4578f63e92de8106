// Matrix products with very few output columns and a long reduction (a softmax-regression
// or classifier head over a handful of rows: [64, 784] x [784, 10]): an MFMA tile would be
// nine tenths padding and ONE workgroup would walk the whole K dimension stage by stage
// (25 stages of fp32, one memory round trip each).  Here every output row is one workgroup of
// one to four wavefronts: thread t takes the 16-byte pieces t, t + threads, .. of the row and of
// every weight row, and the partial sums meet by lane exchanges and, between wavefronts, in LDS.
// fp32 only (the summation order differs from the tiled kernels': within the fp32 bound, as
// theirs differ among themselves).  With every column of a row in one wavefront a Softmax /
// LogSoftmax over the columns is a few more instructions (IgemmParams::row_softmax).
//
// What bounds it is round trips: the rows may lie in page-locked host memory, across PCIe.  So a
// thread requests up to four pieces of its row, and the weights for the first of them, before it
// waits for anything.  64 x 784 x 10 with the rows in host memory: 10.0 us in the kernel trace and
// 27.1 us a call with one wavefront per row, whose turns of one piece each waited for one another;
// 8.4 and 25.2 us now (an empty launch takes 1.9).  From a wavefront per SIMD on (1024 rows: more than the
// room in host memory holds, but for the shortest) the trips hide each other and several wavefronts a row only repeat the lane
// exchanges: there a row keeps one wavefront (rule at the launch).
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>

#include "device_utils.h"
#include "kernels.h"

namespace ohip {
namespace {

// kAhead: pieces of the row a thread requests at once
template <int NB, int NW, int kAhead>
__global__ __launch_bounds__(NW * 64) void gemm_rowdot_kernel(const IgemmParams p) {
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const float* x = reinterpret_cast<const float*>(p.x) + (int64_t)m * p.xcs;
  const float* w = reinterpret_cast<const float*>(p.w);
  float acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) acc[n] = 0.f;
  const int pieces = p.C >> 2;
  for (int k0 = tid; k0 < pieces; k0 += kAhead * NW * 64) {
    floatx4 a[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      // (no piece is requested twice: each is a trip across PCIe where the row is in host memory)
      const int k4 = k0 + u * NW * 64;
      a[u] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (u == 0 || k4 < pieces) a[u] = *reinterpret_cast<const floatx4*>(x + k4 * 4);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int k4 = k0 + u * NW * 64;
      if (k4 >= pieces) break;
      floatx4 b[NB];
      // (columns past the last read the last one's weights: no branch around a request)
#pragma unroll
      for (int n = 0; n < NB; ++n) b[n] = *reinterpret_cast<const floatx4*>(w + (int64_t)(n < p.Kout ? n : p.Kout - 1) * p.w_rs + k4 * 4);
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        acc[n] = __builtin_fmaf(a[u].x, b[n].x, acc[n]);
        acc[n] = __builtin_fmaf(a[u].y, b[n].y, acc[n]);
        acc[n] = __builtin_fmaf(a[u].z, b[n].z, acc[n]);
        acc[n] = __builtin_fmaf(a[u].w, b[n].w, acc[n]);
      }
    }
  }
  // every lane receives every sum of its wavefront; lane n keeps column n
  float mine = 0.f;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const float s = wave_sum(acc[n]);
    mine = lane == n ? s : mine;
  }
  if constexpr (NW > 1) {
    __shared__ float part[NW][16];
    if (lane < NB) part[tid >> 6][lane] = mine;
    __syncthreads();
    if (tid >= 64) return;   // (the first wavefront alone goes on)
    mine = 0.f;
    if (lane < NB) {
#pragma unroll
      for (int q = 0; q < NW; ++q) mine += part[q][lane];
    }
  }
  const bool col = lane < p.Kout;
  const float b = col && p.bias ? reinterpret_cast<const float*>(p.bias)[lane] : 0.f;
  float v = __builtin_fmaf(mine, p.alpha, b);
  v = apply_act(v, p.act, p.act_a, p.act_b);
  if (p.row_softmax != 0) {
    // (wavefront-uniform)  the row's columns sit in lanes 0 .. Kout-1: maximum, exponentials and
    // their sum across the wavefront, the arithmetic of the stand-alone Softmax launch
    const float mx = wave_max(col ? v : -INFINITY);
    const float e = col ? expf(v - mx) : 0.f;
    const float sum = wave_sum(e);
    v = p.row_softmax == 2 ? (v - mx) - logf(sum) : e * (1.0f / sum);
  }
  if (col) reinterpret_cast<float*>(p.y)[(int64_t)m * p.ycs + lane] = v;
}

}  // namespace

bool gemm_rowdot_shape(const IgemmParams& p) {
  if (const char* e = getenv("ODLA_HIP_ROWDOT")) {  // tuning aid: 0 keeps these products on the tiled kernels
    if (e[0] == '0') return false;
  }
  if (const char* force = getenv("ODLA_HIP_IGEMM_TILE")) {
    if (force[0] != 0) return false;
  }
  if (p.in_dt != DT_F32 || p.out_dt != DT_F32) return false;
  if (p.R != 1 || p.S != 1 || p.sh != 1 || p.sw != 1 || p.ph != 0 || p.pw != 0 || p.batch != 1) return false;
  if (p.Ho != p.H || p.Wo != p.W) return false;
  if (p.residual != nullptr || p.y_rdiv > 0 || p.y_zdiv > 0 || p.qmul != nullptr) return false;
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  // few columns, a reduction of at least eight 128-byte stages, and no more rows than keep the
  // weights' re-reads (once per row, out of L2) below the tiled kernel's single pass
  if (p.Kout < 1 || p.Kout > 16 || p.C < 256 || M < 1 || M > 4096) return false;
  if (p.C % 4 != 0 || p.xcs % 4 != 0 || p.w_rs % 4 != 0 || p.w_rs < p.C || p.xcs < p.C || p.ycs < p.Kout) return false;
  return true;
}

hipError_t launch_gemm_rowdot(const IgemmParams& p, hipStream_t stream) {
  auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  if (!gemm_rowdot_shape(p) || p.x == nullptr || p.w == nullptr || p.y == nullptr || !al16(p.x) || !al16(p.w))
    return hipErrorInvalidValue;
  const dim3 grid((unsigned)((int64_t)p.N * p.Ho * p.Wo));
  // As many wavefronts as have pieces, up to four; one request per thread where they reach.  Of many rows one
  // wavefront each, as long as it has at most eight pieces a lane: 16 columns, rows in device memory, several
  // wavefronts / one, us a launch: 1024 rows of 512 5.4 / 5.1, of 1024 7.0 / 6.2, of 2048 9.1 / 8.3; 4096 rows of 1024
  // 13.1 / 11.7; 10 columns, 4096 rows of 784 10.6 / 9.9.  (Longer rows or fewer of them: 1024 of 4096, 10 columns 10.7 /
  // 12.7; 512 of 1024 and 16 columns 5.6 / 5.8.)
  const bool many = grid.x >= 1024 && p.C <= 2048;
#define ROWDOT(NB_)                                                                                              \
  do {                                                                                                           \
    if (many || p.C <= 256) hipLaunchKernelGGL((gemm_rowdot_kernel<NB_, 1, 1>), grid, dim3(64), 0, stream, p);   \
    else if (p.C > 1024) hipLaunchKernelGGL((gemm_rowdot_kernel<NB_, 4, 4>), grid, dim3(256), 0, stream, p);          \
    else if (p.C > 512) hipLaunchKernelGGL((gemm_rowdot_kernel<NB_, 4, 1>), grid, dim3(256), 0, stream, p);      \
    else hipLaunchKernelGGL((gemm_rowdot_kernel<NB_, 2, 1>), grid, dim3(128), 0, stream, p);                     \
  } while (0)
  if (p.Kout <= 4) ROWDOT(4);
  else if (p.Kout <= 8) ROWDOT(8);
  else if (p.Kout <= 12) ROWDOT(12);
  else ROWDOT(16);
#undef ROWDOT
  return hipGetLastError();
}

}  // namespace ohip
