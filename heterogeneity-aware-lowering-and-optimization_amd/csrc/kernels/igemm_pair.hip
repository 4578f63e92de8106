// Two 1x1 layers of 2-byte types in one launch: 64 channels to 128 or 256 (with residual and activation), and those to 64
// or 128 (see IgemmParams::f_y) - the last convolution of a bottleneck block and the first of the next one
// [ref: operators of their own in the reference, ODLA/platforms/dnnl/odla_dnnl.cc].
//
// Both layers are bound by memory, and the wide tensor between them is the largest of the network: 256 images of
// 56 x 56 write 411 MB, which the second layer would read again as a launch of its own.  Here a wavefront takes 32 pixels:
//   - the weights of both layers lie in LDS in fragment order, fetched once by a workgroup that walks the tensor;
//   - 64 channels at a time: the first product, bias, residual and activation in 32 bits, rounded as they are stored; the
//     rounded pixels are the operand of the second product, which adds up over the wide tensor's channels in the
//     order the 128-row tiles of a launch of its own have (results are the same to the bit);
//   - residual in, results out and the operand pass through 4 KiB of LDS of the wavefront (rows of 64 channels,
//     16-byte pieces rotated by the pixel, against bank conflicts), so that memory sees whole 128-byte
//     rows.  No barrier but the one behind the weights.
// A residual that is a layer over 64 channels by itself (the shortcut of a first block) is computed here too, rounded as
// it would be stored: it is neither written nor read.
// The residual of the next two steps and the pixels of the next tile are under way during each step.
// Measured, 64 -> 256 with residual -> 64 / 128 on 256 images of 56 x 56, fp16, two launches and now: 175 + 103 -> 194 - 202
// us (5.2 TB/s over 1.03 GB), 175 + 110 -> 224; with the shortcut's layer 113 + 194 -> 165.  Matrix cores busy 10, 14 and
// 18 % of that time, LDS 27 - 29 % with a fifth to a third of it bank conflicts: neither is what it waits for.
#include "igemm_common.h"
#include "lds_limit.h"

namespace ohip {
namespace {

constexpr int kWaves = 8;
constexpr int kRowsBytes = 32 * 128;                     // 32 pixels x 64 channels

enum { kNoResidual = 0, kResidual = 1, kResidualLayer = 2 };

template <typename T, int N2T, int RES>   // N2T: 32-channel blocks of the second result; RES: the first one's residual
__global__ void __launch_bounds__(kWaves * 64, 2) igemm_pair_kernel(const IgemmParams p, const int tiles) {
  using Acc = typename Mma<T>::Acc;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int n1 = p.Kout, blocks1 = n1 / 32, steps2 = n1 / 16;
  uintx4* w1 = reinterpret_cast<uintx4*>(smem);                         // [block][4][64]
  uintx4* w2 = w1 + blocks1 * 4 * 64;                                   // [block][steps2][64]
  float* b1 = reinterpret_cast<float*>(w2 + N2T * steps2 * 64);
  float* b2 = b1 + n1;
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uintx4* w3 = reinterpret_cast<uintx4*>(b2 + N2T * 32);                // (the residual's layer: as w1 and b1)
  float* b3 = reinterpret_cast<float*>(w3 + (RES == kResidualLayer ? blocks1 * 4 * 64 : 0));
  unsigned char* rows = reinterpret_cast<unsigned char*>(b3 + (RES == kResidualLayer ? n1 : 0)) + wave * kRowsBytes;
  const int M = p.N * p.Ho * p.Wo;

  {
    const uintx4* f1 = reinterpret_cast<const uintx4*>(p.w_frag);
    for (int i = tid; i < blocks1 * 4 * 64; i += kWaves * 64) w1[i] = f1[((i >> 8) * p.wf_chunks + ((i >> 6) & 3)) * 64 + (i & 63)];
    const uintx4* f2 = reinterpret_cast<const uintx4*>(p.f_wfrag);
    for (int j = 0; j < N2T; ++j)
      for (int i = tid; i < steps2 * 64; i += kWaves * 64) w2[j * steps2 * 64 + i] = f2[j * p.f_wf_chunks * 64 + i];
    for (int i = tid; i < n1; i += kWaves * 64) b1[i] = p.bias != nullptr ? reinterpret_cast<const float*>(p.bias)[i] : 0.f;
    for (int i = tid; i < N2T * 32; i += kWaves * 64) b2[i] = p.f_bias != nullptr ? reinterpret_cast<const float*>(p.f_bias)[i] : 0.f;
    if constexpr (RES == kResidualLayer) {
      const uintx4* f3 = reinterpret_cast<const uintx4*>(p.r_wfrag);
      for (int i = tid; i < blocks1 * 4 * 64; i += kWaves * 64) w3[i] = f3[i];
      for (int i = tid; i < n1; i += kWaves * 64) b3[i] = p.r_bias != nullptr ? reinterpret_cast<const float*>(p.r_bias)[i] : 0.f;
    }
  }
  __syncthreads();

  // the wavefronts of a workgroup take neighbouring tiles, workgroups of one XCD neighbouring groups
  int bid = blockIdx.x;
  {
    const int per = gridDim.x >> 3;
    if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
  }
  const int stride = gridDim.x * kWaves;
  auto ordered = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const T* x = reinterpret_cast<const T*>(p.x);
  const T* res = reinterpret_cast<const T*>(p.residual);
  // lane (l32, lg) supplies bytes [32 kk + 16 lg, +16) of pixel l32
  auto load_x = [&](const T* from, const int cs, const int tile, uintx4 (&a)[4]) __attribute__((always_inline)) {
    int m = tile * 32 + l32;
    m = m < M ? m : M - 1;
    const uintx4* row = reinterpret_cast<const uintx4*>(from + (int64_t)m * cs) + lg;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) a[kk] = row[2 * kk];
  };
  // memory side of a row buffer: lane l holds piece l % 8 of pixels l / 8, + 8, ...
  const int piece = lane & 7, px0 = lane >> 3;
  auto load_res = [&](const int tile, const int h, uintx4 (&r)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      int m = tile * 32 + k * 8 + px0;
      m = m < M ? m : M - 1;
      r[k] = *reinterpret_cast<const uintx4*>(res + (int64_t)m * p.rcs + h * 64 + piece * 8);
    }
  };
  unsigned char* mem_at = rows + px0 * 128 + ((piece ^ px0) * 16);       // (pixel k * 8 + px0: k * 1024 behind it)
  auto store_rows = [&](const int tile, T* y, const int cs, const bool stream) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int m = tile * 32 + k * 8 + px0;
      const uintx4 v = *reinterpret_cast<const uintx4*>(mem_at + k * 1024);
      if (m < M) {
        uintx4* d = reinterpret_cast<uintx4*>(y + (int64_t)m * cs + piece * 8);
        if (stream) __builtin_nontemporal_store(v, d);
        else *d = v;
      }
    }
  };
  // accumulator side: lane (l32, lg) holds channels 8 c + 4 lg .. + 3 of pixel l32 for piece c
  auto acc_at = [&](const int c) __attribute__((always_inline)) { return rows + l32 * 128 + ((c ^ (l32 & 7)) * 16) + lg * 8; };

  int tile = bid * kWaves + wave;
  if (tile >= tiles) return;
  // (r0, r1: the residual of two steps; r0: the pixels of its layer)
  uintx4 a[4], a_next[4], r0[4], r1[4];
  load_x(x, p.xcs, tile, a);
  const T* rx = reinterpret_cast<const T*>(p.r_x);
  if constexpr (RES == kResidualLayer) load_x(rx, p.r_xcs, tile, r0);
  if constexpr (RES == kResidual) {
    load_res(tile, 0, r0);
    load_res(tile, 1, r1);
  }
  const int halves = n1 / 64;   // steps of a tile; two or four
  for (; tile < tiles; tile += stride) {
    const int next = tile + stride;
    const int ahead = next < tiles ? next : tile;   // (requested in any case: requests in flight can then be counted)
    load_x(x, p.xcs, ahead, a_next);
    Acc acc2[N2T];
#pragma unroll
    for (int j = 0; j < N2T; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc2[j][e] = 0.f;
    auto step = [&](const int h, auto odd, uintx4 (&r)[4]) __attribute__((always_inline)) {
      if constexpr (RES == kResidual) {
#pragma unroll
        for (int k = 0; k < 4; ++k) *reinterpret_cast<uintx4*>(mem_at + k * 1024) = r[k];
        // the step after the next one, of this tile or the next
        const bool same = h + 2 < halves;
        load_res(same ? tile : ahead, same ? h + 2 : h + 2 - halves, r);
      }
      Acc acc[2];
      uintx2 side[2][4];
      if constexpr (RES == kResidualLayer) {   // the residual's layer, rounded as it would be stored
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[j] = Mma<T>::run(w3[((h * 2 + j) * 4 + kk) * 64 + lane], r0[kk], acc[j]);
        // (the last step requests the next tile's: a second set of registers would not fit)
        if constexpr (decltype(odd)::value) load_x(rx, p.r_xcs, h + 1 < halves ? tile : ahead, r0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const floatx4 b = *reinterpret_cast<const floatx4*>(b3 + h * 64 + j * 32 + q * 8 + lg * 4);
            const Acc& v = acc[j];
            side[j][q] = uintx2{pack2<T>(v[q * 4] + b.x, v[q * 4 + 1] + b.y), pack2<T>(v[q * 4 + 2] + b.z, v[q * 4 + 3] + b.w)};
          }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = Mma<T>::run(w1[((h * 2 + j) * 4 + kk) * 64 + lane], a[kk], acc[j]);
      ordered();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          unsigned char* at = acc_at(j * 4 + q);
          const floatx4 b = *reinterpret_cast<const floatx4*>(b1 + h * 64 + j * 32 + q * 8 + lg * 4);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[j][q * 4 + e] + b[e];
          if constexpr (RES != kNoResidual) {
            const uintx2 t = RES == kResidualLayer ? side[j][q] : *reinterpret_cast<const uintx2*>(at);
            const T* rt = reinterpret_cast<const T*>(&t);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += Store<T>::ld(rt + e);
          }
          if (p.act == ACT_RELU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
          }
          *reinterpret_cast<uintx2*>(at) = uintx2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        }
      ordered();
      store_rows(tile, reinterpret_cast<T*>(p.y) + h * 64, p.ycs, p.stream_out);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const uintx4 o = *reinterpret_cast<const uintx4*>(rows + l32 * 128 + (((2 * kk + lg) ^ (l32 & 7)) * 16));
#pragma unroll
        for (int j = 0; j < N2T; ++j) acc2[j] = Mma<T>::run(w2[(j * steps2 + h * 4 + kk) * 64 + lane], o, acc2[j]);
      }
      ordered();
    };
#pragma unroll 1
    for (int h = 0; h < halves; h += 2) {
      step(h, std::false_type(), r0);
      step(h + 1, std::true_type(), r1);
    }
    // the second result, 64 channels at a time
#pragma unroll
    for (int g = 0; g < N2T / 2; ++g) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 b = *reinterpret_cast<const floatx4*>(b2 + g * 64 + j * 32 + q * 8 + lg * 4);
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc2[g * 2 + j][q * 4 + e] + b[e];
            if (p.f_act == ACT_RELU) v[e] = v[e] > 0.f ? v[e] : 0.f;
          }
          *reinterpret_cast<uintx2*>(acc_at(j * 4 + q)) = uintx2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        }
      ordered();
      store_rows(tile, reinterpret_cast<T*>(p.f_y) + g * 64, p.f_ycs, false);
      ordered();
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      a[kk] = a_next[kk];
    }
  }
}

// Where one launch is the faster form.  The 2048 wavefronts of the launch take one tile each up to 2^16 pixels.
// Measured as four blocks of a first stage (3x3 layers and pairs, a mean behind them), fp16, launches apart / one launch,
// n images of 3136 pixels: 64 -> 256 -> 64, 64 -> 256 -> 128, 64 -> 128 -> 64, 64 -> 256 -> 64 with the shortcut's layer:
//   n = 2: 111 / 126, 122 / 144, 102 / 108, 112 / 125 us   (fetch of the weights and one tile's chain of latencies)
//   8: 158 / 163, 175 / 177, 134 / 138, 161 / 160     10: 161 / 164, 176 / 183, 144 / 143, 162 / 156
//   14: 204 / 190, 219 / 214, 179 / 168, 206 / 178    20: 241 / 213, 273 / 246, 200 / 189, 242 / 198
//   21: 247 / 242, 289 / 292, 209 / 209, 248 / 227    26: 264 / 256, 318 / 308, 217 / 217, 267 / 245
//   28: 279 / 267, 329 / 317, 230 / 226, 282 / 256    40: 343 / 310, 407 / 366, 273 / 251, 342 / 288
//   64: 473 / 420, 617 / 588, 364 / 327, 475 / 396    128: 903 / 808, 1156 / 1018, 614 / 572, 910 / 757
// Below 2^15 pixels only the form with the shortcut's layer gains, which is not known yet when the pair is (all of
// ResNet-50 fp16, which has one of these among its three pairs, at 8 images: 492 / 478).  Between one and 1.3 tiles a
// wavefront little is gained alone, and more is lost where two halves of a batch run side by side: all of ResNet-50 fp16,
// halves of 22 images 966 / 1020, of 24 1028 / 1052, of 26 1085 / 1094, of 28 1155 / 1145, of 30 1207 / 1189, of 36 1366 / 1311,
// of 48 1685 / 1631 (and of 20 920 / 938, where 20 images alone take 655 / 622).
constexpr int64_t kPairPixels = 1 << 15, kOneTile = 64 << 10, kTwoTiles = 84 << 10;
bool pair_pays(const int64_t pixels) {
  if (const char* e = getenv("ODLA_HIP_PAIR_MIN_PIXELS")) return pixels >= atoll(e);   // test aid
  return pixels >= kPairPixels && (pixels <= kOneTile || pixels >= kTwoTiles);
}

constexpr int pair_lds(const int n1, const int n2, const bool layer) { return n1 * (layer ? 256 : 128) + n2 * n1 * 2 + (n1 * (layer ? 2 : 1) + n2) * 4 + kWaves * kRowsBytes; }
constexpr int kMostLds = pair_lds(256, 64, true) > pair_lds(256, 128, false) ? pair_lds(256, 64, true) : pair_lds(256, 128, false);
static_assert(kMostLds <= 160 * 1024, "LDS of a compute unit");

template <typename T>
hipError_t launch_typed(const IgemmParams& p, hipStream_t stream) {
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  const int tiles = (int)((M + 31) / 32);
  const int lds = pair_lds(p.Kout, p.f_kout, p.r_x != nullptr);
  int grid = (tiles + kWaves - 1) / kWaves;
  if (grid > 256) grid = 256;
  auto go = [&](auto kernel, LdsLimit& limit) -> hipError_t {
    const hipError_t e = limit.raise(reinterpret_cast<const void*>(kernel), kMostLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kWaves * 64), (size_t)lds, stream, p, tiles);
    return hipGetLastError();
  };
  static LdsLimit limits[5];   // (of this type's instances, in the order below)
  if (p.r_x != nullptr) return go(igemm_pair_kernel<T, 2, kResidualLayer>, limits[0]);
  if (p.residual != nullptr) return p.f_kout == 64 ? go(igemm_pair_kernel<T, 2, kResidual>, limits[1]) : go(igemm_pair_kernel<T, 4, kResidual>, limits[2]);
  return p.f_kout == 64 ? go(igemm_pair_kernel<T, 2, kNoResidual>, limits[3]) : go(igemm_pair_kernel<T, 4, kNoResidual>, limits[4]);
}

}  // namespace

namespace {
bool pointwise(const IgemmParams& p) {
  return p.R == 1 && p.S == 1 && p.sh == 1 && p.sw == 1 && p.ph == 0 && p.pw == 0 && p.batch == 1 && p.Ho == p.H && p.Wo == p.W &&
         p.alpha == 1.f && (p.act == ACT_NONE || p.act == ACT_RELU) && p.y_rdiv == 0 && p.row_softmax == 0 && !p.ln && p.f_y == nullptr &&
         p.wf_chunks * 16 == p.C;
}
}  // namespace

// a: the wide layer, b: the one that reads its result; no pointer is looked at.
bool igemm_pair_fusable(const IgemmParams& a, const IgemmParams& b) {
  if ((a.in_dt != DT_F16 && a.in_dt != DT_BF16) || a.out_dt != a.in_dt || b.in_dt != a.in_dt || b.out_dt != a.in_dt) return false;
  if (!pointwise(a) || !pointwise(b) || a.res_after_act) return false;
  if (a.C != 64 || (a.Kout != 128 && a.Kout != 256) || a.ycs != a.Kout || a.xcs % 8 != 0) return false;
  if (b.C != a.Kout || b.xcs != a.ycs || (b.Kout != 64 && b.Kout != 128) || b.ycs % 8 != 0) return false;
  if (b.N != a.N || b.H != a.Ho || b.W != a.Wo) return false;
  const int64_t M = (int64_t)a.N * a.Ho * a.Wo;
  return M < (1ll << 30) && pair_pays(M);
}

// r: the layer whose result is the residual of a (f_kout channels behind), and nothing else reads.
bool igemm_pair_residual(const IgemmParams& a, const int f_kout, const IgemmParams& r) {
  return f_kout == 64 && pointwise(r) && r.act == ACT_NONE && r.in_dt == a.in_dt && r.out_dt == a.in_dt && r.C == 64 && r.Kout == a.Kout && r.ycs == r.Kout && r.xcs % 8 == 0 &&
         r.N == a.N && r.H == a.H && r.W == a.W;   // (128 channels behind: three sets of weights do not fit)
}

hipError_t launch_igemm_pair(const IgemmParams& p, hipStream_t stream) {
  auto al16 = [](const void* q) { return q != nullptr && (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  if (p.C != 64 || (p.Kout != 128 && p.Kout != 256) || (p.f_kout != 64 && p.f_kout != 128) || p.wf_chunks != 4 || p.f_wf_chunks * 16 != p.Kout) return hipErrorInvalidValue;
  if (!al16(p.x) || !al16(p.y) || !al16(p.f_y) || !al16(p.w_frag) || !al16(p.f_wfrag) || (p.residual != nullptr && !al16(p.residual))) return hipErrorInvalidValue;
  if (p.xcs % 8 != 0 || p.ycs != p.Kout || p.f_ycs % 8 != 0 || p.f_ycs < p.f_kout || (p.residual != nullptr && (p.rcs % 8 != 0 || p.rcs < p.Kout))) return hipErrorInvalidValue;
  if (p.r_x != nullptr && (p.residual != nullptr || !al16(p.r_x) || !al16(p.r_wfrag) || p.r_xcs % 8 != 0 || p.r_xcs < 64 || p.f_kout != 64)) return hipErrorInvalidValue;
  if ((int64_t)p.N * p.Ho * p.Wo <= 0 || (int64_t)p.N * p.Ho * p.Wo >= (1ll << 30)) return hipErrorInvalidValue;
  return p.in_dt == DT_F16 ? launch_typed<f16_t>(p, stream) : p.in_dt == DT_BF16 ? launch_typed<bf16_t>(p, stream) : hipErrorInvalidValue;
}

}  // namespace ohip
