// Implicit GEMM for launches with few output tiles: batch-1 .. batch-16 images, single
// sequences, the small feature maps at the end of a network.
//
// What bounds such a launch is not bandwidth or the matrix cores but one workgroup's chain of
// K stages (128-pixel x 128-channel tiles: ResNet-50's last 3x3 layer at one image is four
// workgroups of 72 stages, 32 us) on a mostly idle chip.  Here
//   - the output tile is small (16 x 16 or 32 x 32 pixels x channels, 16x16 MFMA blocks), so that
//     a layer of 49 pixels x 512 channels is 128 workgroups instead of four;
//   - the wavefronts of a workgroup (16 or 8 of them) all own the SAME tile and split K: each walks a
//     contiguous share of the 64-byte K steps, so the chain is a few steps long and its loads
//     are all in flight together;
//   - both operands go straight from global memory into MFMA registers (16 bytes per lane; the
//     caches serve what workgroups share), no staging, no barrier in the K loop;
//   - the partial tiles are added through LDS in a fixed order by the threads that then apply
//     the epilogue to four consecutive channels of one pixel each.
// Any tap geometry, stride, dilation, padding, grid.z batch and operand type of IgemmParams is
// served; weights are read from the fragment-ordered copy where one exists, from the packed
// rows otherwise.
//
// Where a launch's 4 .. 9 us go (clock stamps, chains of captured launches): 1.3 us between the
// last store of a launch and the first instruction of the next, 0.4 - 0.6 us arguments and
// addresses, 0.6 us the last store, 0.2 - 0.5 us the start of all workgroups, and the rest is the
// K loop, which is its round trips to memory and, from some 100 KB per workgroup on, the 64 bytes
// per clock of a compute unit's L1.  Hence all requests of up to 2 U steps at once, with nothing
// behind a request that waits for it: as two or four steps at a time, with the select of padding
// lanes right behind each request (a wait), 14 x 14 maps of one image took 6.3 (3x3 256 -> 256) and
// 5.1 us (1x1 1024 -> 256) with the 16-wide tile, and take 6.0 and 4.5; ResNet-50 fp16 at one image
// 316 -> 302 us, fp32 at four images from host arrays 973 -> 853 us, BERT-base bf16 at 1 x 41 tokens 400 -> 389 us.
//
// A LayerNorm in front of a product of so few rows is a launch of 4 us for 60 KB, beside a
// product that reads every row whole in each of its workgroups anyway: SLIM_LN takes it along.
// A wavefront holds its share of K of the 16 or 32 rows in registers (at most three steps), the
// rows' sums and then their squared deviations meet in LDS, and the normalised values, rounded as
// the stand-alone launch rounds them, are the operand; the workgroups of the first channel tile
// also write them for whoever else reads the result.  BERT-base bf16 at 1 x 41 tokens: 24 of 91
// launches less.
#include "igemm_common.h"

#include <cstdlib>
#include <cstring>

namespace ohip {

// 16x16 blocks: lane l feeds row l % 16 of either operand with the 16 bytes l / 16 of a 64-byte
// K step, and ends up with four consecutive channels ((l / 16) * 4 ..) of pixel l % 16.
template <typename T> struct Mma16;
template <> struct Mma16<float> {
  using Acc = floatx4;
  __device__ static __forceinline__ Acc run(uintx4 a, uintx4 b, Acc c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
    return c;
  }
};
template <> struct Mma16<f16_t> {
  using Acc = floatx4;
  __device__ static __forceinline__ Acc run(uintx4 a, uintx4 b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  }
};
template <> struct Mma16<bf16_t> {
  using Acc = floatx4;
  __device__ static __forceinline__ Acc run(uintx4 a, uintx4 b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma16<int8_t> {
  using Acc = intx4;
  __device__ static __forceinline__ Acc run(uintx4 a, uintx4 b, Acc c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(intx4, a), __builtin_bit_cast(intx4, b), c, 0, 0, 0);
  }
};

// What the launcher works out once per launch.
struct SlimArgs {
  int tiles_m = 0, tiles_n = 0;
  int m_fast = 0;        // neighbouring workgroups share channels (1) or pixels (0)
  int t_div = 1, t_shift = 0;   // division of a workgroup's number by the tiles of the fast direction
  unsigned t_magic = 0;
  int steps = 0;         // 64-byte K steps, the last one possibly partial
  int cvec = 1;          // 16-byte vectors per tap
  unsigned cv_magic = 0, s_magic = 0;
  int cv_shift = 0, s_shift = 0;
};

// How K maps to taps: one contiguous run per pixel / a step inside one tap / any.
enum SlimMode { SLIM_ROW = 0, SLIM_TAP = 1, SLIM_ANY = 2,
                SLIM_LN = 3,     // one run per pixel, normalised: rows of the operand's type
                SLIM_LN32 = 4 }; // ... rows of floats under a 2-byte operand
constexpr int kSlimLnSteps = 3;   // K steps of a wavefront it can hold

// 16 bytes at byte `off` of a buffer; zero where off is kNoByte.  (A lane without a pixel or behind
// the end of K needs no select on the loaded value then: such a select is a wait for the value, and
// the compiler puts it next to the request.)
constexpr unsigned kNoByte = 0xffffffffu;
#if defined(__HIP_DEVICE_COMPILE__)  // (the builtins are unknown to the host pass, which only needs the launch stub)
using SlimBuf = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ SlimBuf slim_buf(const unsigned char* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(base), 0, 0x7fffffff, 0x00020000);
}
__device__ __forceinline__ uintx4 slim_load(const SlimBuf b, const unsigned off, const unsigned soff) {
  return __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(b, (int)off, (int)soff, 0));
}
#else
using SlimBuf = const unsigned char*;
__device__ __forceinline__ SlimBuf slim_buf(const unsigned char* base) { return base; }
__device__ __forceinline__ uintx4 slim_load(const SlimBuf, const unsigned, const unsigned) { return uintx4{0, 0, 0, 0}; }
#endif

template <typename TIn, typename Epi, int MB, int NB, int NW, int MODE>
__global__ void __launch_bounds__(NW * 64, 4)
igemm_slim_kernel(const IgemmParams p, const int epi_vec, const SlimArgs a) {
  using Acc = typename Mma16<TIn>::Acc;
  using AccE = typename Epi::AccE;
  using TOut = typename EpiTraits<Epi>::TOut;
  typedef AccE accx4 __attribute__((ext_vector_type(4)));
  constexpr int ES = sizeof(TIn);
  constexpr int BM = MB * 16, BN = NB * 16;
  constexpr int PITCH = BN + 4;             // words per pixel of a partial tile
  constexpr int U = MB + NB <= 2 ? 5 : ES == 1 && MODE == SLIM_ANY ? 1 : MODE == SLIM_ANY || (ES == 1 && MODE == SLIM_TAP) ? 2 : 3;   // K steps of a batch; two batches are in flight
  constexpr int REGION = BM * PITCH * 4;    // bytes of a wavefront's partial tile
  constexpr int UNITS = BM * BN / 4;        // (pixel, four channels) pairs of the tile
  constexpr int UPT = (UNITS + NW * 64 - 1) / (NW * 64);
  static_assert(UNITS % 64 == 0, "whole wavefronts in the epilogue");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  fetch_args(p.x, p.w, p.w_frag, p.wf_chunks, p.wf_tiles, p.N, p.H, p.W, p.C, p.xcs, p.Ho, p.Wo, p.sh, p.sw, p.ph, p.pw, p.howo_magic,
             p.howo_shift, p.wo_magic, p.wo_shift, p.x_bs, a.tiles_m, a.tiles_n, a.m_fast, a.t_div, a.t_shift, a.t_magic, a.steps, a.cvec, p.Kout, p.w_bs, p.w_rs, p.w_rows);
  if constexpr (MODE == SLIM_LN || MODE == SLIM_LN32) fetch_args(p.ln_x, p.ln_g, p.ln_b, p.ln_y, p.ln_eps);
  fetch_args(p.bias, p.residual, p.y, p.ycs, p.rcs, p.y_bs, p.y_rdiv, p.y_zdiv, p.alpha, p.act, p.act_a, p.act_b, epi_vec);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int M = p.N * p.Ho * p.Wo;
  // workgroups that share operands stay on one XCD (they are dealt round-robin)
  int bid = blockIdx.x;
  {
    const int per = (a.tiles_m * a.tiles_n) >> 3;   // (gridDim is a load of its own)
    if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
  }
  const int outer = fast_div(bid, a.t_magic, a.t_shift), inner = bid - outer * a.t_div;
  const int tile_m = a.m_fast ? inner : outer;
  const int tile_n = a.m_fast ? outer : inner;
  const int z = blockIdx.z;

  // ---- this wavefront's share of the K steps ----
  const int per = a.steps / NW, extra = a.steps - per * NW;
  const int k0 = wave * per + (wave < extra ? wave : extra);
  const int k1 = k0 + per + (wave < extra ? 1 : 0);
  const int kvecs = p.R * p.S * a.cvec;          // valid 16-byte vectors of K

  // ---- weights: scalar base, a lane's bytes from there, bytes per 64 bytes of K ----
  SlimBuf w_buf[NB];
  unsigned w_off[NB];
  const bool frag = p.w_frag != nullptr;
  const int w_step = frag ? 2048 : 64;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n0 = tile_n * BN + j * 16;
    const unsigned char* base;
    if (frag) {
      int t = n0 >> 5;
      t = t < p.wf_tiles ? t : p.wf_tiles - 1;   // surplus channels are computed and never stored
      base = reinterpret_cast<const unsigned char*>(p.w_frag) + ((int64_t)z * p.wf_tiles + t) * p.wf_chunks * 1024;
      w_off[j] = (unsigned)((g >> 1) * 1024 + ((g & 1) * 32 + ((n0 + l16) & 31)) * 16);
    } else {
      const int r0 = n0 < p.w_rows ? n0 : p.w_rows - 1, r = n0 + l16 < p.w_rows ? n0 + l16 : p.w_rows - 1;
      base = reinterpret_cast<const unsigned char*>(reinterpret_cast<const TIn*>(p.w) + (int64_t)z * p.w_bs + (int64_t)r0 * p.w_rs);
      w_off[j] = (unsigned)((r - r0) * p.w_rs * ES + g * 16);
    }
    w_buf[j] = slim_buf(base);
  }
  auto load_w = [&](const int k, uintx4 (&W)[NB]) __attribute__((always_inline)) {
    // (packed rows end at w_cols: the last step may reach behind them)
    const bool in = MODE == SLIM_TAP || k * 4 + g < kvecs;
#pragma unroll
    for (int j = 0; j < NB; ++j) W[j] = slim_load(w_buf[j], in ? w_off[j] : kNoByte, (unsigned)(k * w_step));
  };

  // ---- pixels: scalar base (the tile's first image), a lane's bytes from there at tap (0, 0), channel 0 ----
  const int HoWo = p.Ho * p.Wo;
  const int img_bytes = p.H * p.W * p.xcs * ES;
  const int img0 = fast_div(tile_m * BM, p.howo_magic, p.howo_shift);
  const SlimBuf x_buf = slim_buf(reinterpret_cast<const unsigned char*>(reinterpret_cast<const TIn*>(p.x) + (int64_t)z * p.x_bs) + (int64_t)img0 * img_bytes);
  int a_off[MB], a_hi[MB], a_wi[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    int m = tile_m * BM + i * 16 + l16;
    m = m < M ? m : M - 1;                       // surplus rows are computed and never stored
    const int n_img = fast_div(m, p.howo_magic, p.howo_shift);
    const int rem = m - n_img * HoWo;
    const int ho = fast_div(rem, p.wo_magic, p.wo_shift);
    const int wo = rem - ho * p.Wo;
    a_hi[i] = ho * p.sh - p.ph;
    a_wi[i] = wo * p.sw - p.pw;
    a_off[i] = (n_img - img0) * img_bytes + (a_hi[i] * p.W + a_wi[i]) * p.xcs * ES + (MODE == SLIM_ANY ? 0 : g * 16);
  }

  // walk of SLIM_TAP: wavefront-uniform tap and step inside the tap
  int kc = 0, kr = 0, ks = 0;
  const int cps = a.cvec >> 2;
  if constexpr (MODE == SLIM_TAP) {
    const int tap = fast_div(k0 * 4, a.cv_magic, a.cv_shift);
    kc = k0 - tap * cps;
    kr = fast_div(tap, a.s_magic, a.s_shift);
    ks = tap - kr * p.S;
  }
  // Padding taps of 8-bit operands hold the stored byte of the value 0, which no load returns by
  // itself: those lanes keep a mask for the select at the use.
  constexpr bool kFill = ES == 1 && MODE != SLIM_ROW;
  const unsigned f = (unsigned)(p.a_fill & 0xff) * 0x01010101u;
  auto load_a = [&](const int k, uintx4 (&A)[MB], bool (&okv)[MB]) __attribute__((always_inline)) {
    if constexpr (MODE == SLIM_ROW) {
      const bool in = k * 4 + g < kvecs;
#pragma unroll
      for (int i = 0; i < MB; ++i) A[i] = slim_load(x_buf, in ? (unsigned)(a_off[i] + k * 64) : kNoByte, 0u);
    } else {
      int hoff, woff, coff;
      bool in = true;
      if constexpr (MODE == SLIM_TAP) {
        hoff = kr * p.dh; woff = ks * p.dw; coff = kc * 64;
        const int tap_end = ++kc == cps ? 1 : 0;
        kc = tap_end ? 0 : kc;
        ks += tap_end;
        const int row_end = ks == p.S ? 1 : 0;
        ks = row_end ? 0 : ks;
        kr += row_end;
      } else {
        const int kv = k * 4 + g;
        in = kv < kvecs;
        const int tap = fast_div(kv, a.cv_magic, a.cv_shift);
        const int r = fast_div(tap, a.s_magic, a.s_shift);
        hoff = r * p.dh; woff = (tap - r * p.S) * p.dw; coff = (kv - tap * a.cvec) * 16;
      }
      const int off = (hoff * p.W + woff) * p.xcs * ES + coff;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const bool ok = in && (unsigned)(a_hi[i] + hoff) < (unsigned)p.H && (unsigned)(a_wi[i] + woff) < (unsigned)p.W;
        A[i] = slim_load(x_buf, ok ? (unsigned)(a_off[i] + off) : kNoByte, 0u);
        if constexpr (kFill) okv[i] = ok;
      }
    }
  };

  Acc acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = Acc{0, 0, 0, 0};
  auto mul = [&](const uintx4 (&A)[MB], const uintx4 (&W)[NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = Mma16<TIn>::run(W[j], A[i], acc[i][j]);
  };
  // U steps at once: requested together, multiplied together
  struct Batch {
    uintx4 A[U][MB], W[U][NB];
    bool ok[U][MB];
  };
  auto load = [&](const int at, auto count, Batch& b) __attribute__((always_inline)) {
    constexpr int n = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < n; ++u) { load_w(at + u, b.W[u]); load_a(at + u, b.A[u], b.ok[u]); }
  };
  auto use = [&](auto count, Batch& b) __attribute__((always_inline)) {
    constexpr int n = decltype(count)::value;
#pragma unroll
    for (int u = 0; u < n; ++u) {
      if constexpr (kFill) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          asm volatile("" : "+v"(b.A[u][i]));   // the select belongs here, not to the request
          b.A[u][i] = b.ok[u][i] ? b.A[u][i] : uintx4{f, f, f, f};
        }
      }
      mul(b.A[u], b.W[u]);
    }
  };

  // ---- operands of the epilogue: requested behind the first batch, so that they travel with it ----
  const AccE* bias = p.bias ? reinterpret_cast<const AccE*>(p.bias) + (int64_t)z * p.bias_bs : nullptr;
  TOut* ybase = reinterpret_cast<TOut*>(p.y) + (EpiTraits<Epi>::quant ? (int64_t)z * p.y_bs : y_batch_off(p, z));
  const TOut* rbase = p.residual ? reinterpret_cast<const TOut*>(p.residual) + (int64_t)z * p.r_bs : nullptr;
  constexpr bool kQ8 = std::is_same<Epi, EpiQuant<0>>::value;
  const bool wide = (epi_vec & 1) != 0;
  // raw: a conversion here would be a wait for the request here
  uintx4 b_raw[UPT], m_raw[UPT];
  typename std::conditional<sizeof(TOut) == 4, uintx4, typename std::conditional<sizeof(TOut) == 2, uintx2, unsigned>::type>::type r_raw[UPT];
  const bool q_wide = EpiTraits<Epi>::quant && p.qmul != nullptr && (reinterpret_cast<uintptr_t>(p.qmul) & 15u) == 0;
  auto fetch_epi = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < UPT; ++t) {
      const int u = tid + t * NW * 64;
      const int m = tile_m * BM + u / (BN / 4), n = tile_n * BN + (u % (BN / 4)) * 4;
      if (u < UNITS && m < M && wide && n + 4 <= p.Kout) {
        if (bias != nullptr) b_raw[t] = *reinterpret_cast<const uintx4*>(bias + n);
        if (rbase != nullptr) __builtin_memcpy(&r_raw[t], __builtin_assume_aligned(rbase + (int64_t)m * p.rcs + n, sizeof(TOut) * 4), sizeof(TOut) * 4);
        if constexpr (EpiTraits<Epi>::quant) {
          if (q_wide) m_raw[t] = *reinterpret_cast<const uintx4*>(p.qmul + n);
        }
      }
    }
  };

  if constexpr (MODE == SLIM_LN || MODE == SLIM_LN32) {
    constexpr int LU = kSlimLnSteps, E = 16 / ES;   // elements of a lane per step
    using TX = typename std::conditional<MODE == SLIM_LN32, float, TIn>::type;
    __shared__ float ln_sum[2][NW][BM];
    __shared__ __attribute__((aligned(16))) float ln_gb[2][LU * NW * 4 * E];
    // scale and offset of all channels: a piece or two per thread, requested first, in LDS behind
    // the other requests and ahead of the first barrier
    constexpr int GBH = LU * NW * 4 * E, GBR = (2 * GBH / 4 + NW * 64 - 1) / (NW * 64);
    floatx4 gbv[GBR];
#pragma unroll
    for (int r = 0; r < GBR; ++r) {
      const int c = tid * 4 + r * NW * 256, which = c >= GBH, cc = c - which * GBH;
      const float* src = which ? p.ln_b : p.ln_g;
      const float d = which ? 0.f : 1.f;
      const bool in = src != nullptr && cc < p.C;
      const floatx4 got = *reinterpret_cast<const floatx4*>(in ? src + cc : reinterpret_cast<const float*>(p.ln_x));
      gbv[r] = in ? got : floatx4{d, d, d, d};
    }
    const int cnt = k1 - k0;                        // 1 .. LU, the same for a whole wavefront
    uintx4 W[LU][NB];
    float v[LU][MB][E];
    const TX* lx = reinterpret_cast<const TX*>(p.ln_x);
    int64_t at[MB];                                 // element of this lane's first piece, per row
    bool live[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int m = tile_m * BM + i * 16 + l16;
      live[i] = m < M;
      at[i] = (int64_t)(m < M ? m : M - 1) * p.C + g * E;
    }
    // (steps past the wavefront's share repeat its last one and are left out of the sums)
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int k = u < cnt ? k0 + u : k1 - 1;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        constexpr int VX = 16 / sizeof(TX);
#pragma unroll
        for (int h = 0; h < E / VX; ++h) {
          Vec16<TX> t;
          t.load(lx + at[i] + k * (4 * E) + h * VX);
#pragma unroll
          for (int e = 0; e < VX; ++e) v[u][i][h * VX + e] = t.get(e);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int k = u < cnt ? k0 + u : k1 - 1;
      load_w(k, W[u]);
    }
#pragma unroll
    for (int r = 0; r < GBR; ++r) {
      const int c = tid * 4 + r * NW * 256;
      if (c < 2 * GBH) *reinterpret_cast<floatx4*>(&ln_gb[0][0] + c) = gbv[r];
    }
    float mean[MB], rstd[MB];
    // the four lanes of a row, then the wavefronts
    auto row_sums = [&](const int which, float (&s)[MB]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        s[i] += __shfl_xor(s[i], 16);
        s[i] += __shfl_xor(s[i], 32);
        if (g == 0) ln_sum[which][wave][i * 16 + l16] = s[i];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        s[i] = ln_sum[which][0][i * 16 + l16];
#pragma unroll
        for (int w = 1; w < NW; ++w) s[i] += ln_sum[which][w][i * 16 + l16];
      }
    };
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      mean[i] = 0.f;
#pragma unroll
      for (int u = 0; u < LU; ++u) {
        if (u >= cnt) break;
#pragma unroll
        for (int e = 0; e < E; ++e) mean[i] += v[u][i][e];
      }
    }
    row_sums(0, mean);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      mean[i] /= (float)p.C;
      rstd[i] = 0.f;
#pragma unroll
      for (int u = 0; u < LU; ++u) {
        if (u >= cnt) break;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          v[u][i][e] -= mean[i];
          rstd[i] = __builtin_fmaf(v[u][i][e], v[u][i][e], rstd[i]);
        }
      }
    }
    row_sums(1, rstd);
    if constexpr (MB == 1) fetch_epi();   // (at 32 rows there are no registers for them here)
#pragma unroll
    for (int i = 0; i < MB; ++i) rstd[i] = 1.0f / sqrtf(rstd[i] / (float)p.C + p.ln_eps);
    const bool writes = tile_n == 0 && z == 0;
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      if (u >= cnt) break;
      const int e0 = (k0 + u) * (4 * E);
      float ga[E], be[E];
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        const floatx4 gv = *reinterpret_cast<const floatx4*>(&ln_gb[0][e0 + g * E + e]);
        const floatx4 bv = *reinterpret_cast<const floatx4*>(&ln_gb[1][e0 + g * E + e]);
#pragma unroll
        for (int q = 0; q < 4; ++q) { ga[e + q] = gv[q]; be[e + q] = bv[q]; }
      }
      uintx4 A[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        float o[E];
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] = __builtin_fmaf(v[u][i][e] * rstd[i], ga[e], be[e]);
        if constexpr (ES == 4) A[i] = __builtin_bit_cast(uintx4, floatx4{o[0], o[1], o[2], o[3]});
        else A[i] = uintx4{pack2<TIn>(o[0], o[1]), pack2<TIn>(o[2], o[3]), pack2<TIn>(o[4], o[5]), pack2<TIn>(o[6], o[7])};
        if (writes && live[i]) {
          if constexpr (MODE == SLIM_LN32) {
            float* y = reinterpret_cast<float*>(p.ln_y) + at[i] + e0;
#pragma unroll
            for (int e = 0; e < E; e += 4) *reinterpret_cast<floatx4*>(y + e) = floatx4{o[e], o[e + 1], o[e + 2], o[e + 3]};
            if (p.ln_y2 != nullptr) *reinterpret_cast<uintx4*>(reinterpret_cast<TIn*>(p.ln_y2) + at[i] + e0) = A[i];
          } else {
            *reinterpret_cast<uintx4*>(reinterpret_cast<TIn*>(p.ln_y) + at[i] + e0) = A[i];
          }
        }
      }
      mul(A, W[u]);
    }
    if constexpr (MB > 1) fetch_epi();
  } else {
    // Straight-line code for every number of steps up to 2 U: all of them are in flight together.
    // Longer shares: a full batch and what fills none first, then full batches in turn, the next one
    // requested before the one in hand is multiplied.  (Requests in conditional code cannot be
    // counted: the compiler would wait for all of them at every use.)
    constexpr std::integral_constant<int, U> full{};
    Batch b0, b1;
    const int n = k1 - k0, batches = n / U, rest = n - batches * U;
    if (batches == 0) {
      static_for<U>([&](auto r) __attribute__((always_inline)) {   // (no steps: the epilogue's operands all the same)
        if (rest != decltype(r)::value) return;
        load(k0, r, b0);
        fetch_epi();
        use(r, b0);
      });
    } else {
      static_for<U>([&](auto r) __attribute__((always_inline)) {
        if (rest != decltype(r)::value) return;
        load(k0, r, b0);
        load(k0 + decltype(r)::value, full, b1);
        fetch_epi();
        use(r, b0);
      });
      int k = k0 + rest;   // b1 holds the batch at k
      for (; k + 3 * U <= k1; k += 2 * U) {
        load(k + U, full, b0);
        use(full, b1);
        load(k + 2 * U, full, b1);
        use(full, b0);
      }
      if (k + 2 * U <= k1) {
        load(k + U, full, b0);
        use(full, b1);
        use(full, b0);
      } else {
        use(full, b1);
      }
    }
  }

  unsigned char* mine = smem + wave * REGION;
  // ---- partial tiles through LDS ----
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
      *reinterpret_cast<accx4*>(reinterpret_cast<AccE*>(mine) + (i * 16 + l16) * PITCH + j * 16 + g * 4) = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < UPT; ++t) {
    const int u = tid + t * NW * 64;
    const int pix = u / (BN / 4), c = (u % (BN / 4)) * 4;
    const int m = tile_m * BM + pix, n = tile_n * BN + c;
    if (u >= UNITS || m >= M || n >= p.Kout) continue;
    accx4 s = *reinterpret_cast<const accx4*>(smem + (pix * PITCH + c) * 4);
#pragma unroll
    for (int w = 1; w < NW; ++w) s += *reinterpret_cast<const accx4*>(smem + w * REGION + (pix * PITCH + c) * 4);
    const bool vec = wide && n + 4 <= p.Kout;
    AccE b4[4] = {0, 0, 0, 0};
    float m4[4] = {0.f, 0.f, 0.f, 0.f}, r4[4] = {0.f, 0.f, 0.f, 0.f};
    unsigned rq = 0u;
    if (vec) {
      if (bias != nullptr) __builtin_memcpy(b4, &b_raw[t], 16);
      if (rbase != nullptr) {
        if constexpr (kQ8) rq = r_raw[t];
        else {
          TOut e4[4];
          __builtin_memcpy(e4, &r_raw[t], sizeof(e4));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (sizeof(TOut) == 4) r4[e] = (float)e4[e];
            else r4[e] = Store<TOut>::ld(e4 + e);
          }
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= p.Kout) break;
        if (bias != nullptr) b4[e] = bias[n + e];
        if (rbase != nullptr) {
          if constexpr (kQ8) rq |= (unsigned)(uint8_t)rbase[(int64_t)m * p.rcs + n + e] << (8 * e);
          else if constexpr (sizeof(TOut) == 4) r4[e] = (float)rbase[(int64_t)m * p.rcs + n + e];
          else r4[e] = Store<TOut>::ld(rbase + (int64_t)m * p.rcs + n + e);
        }
      }
    }
    if constexpr (EpiTraits<Epi>::quant) {
      if (vec && q_wide) __builtin_memcpy(m4, &m_raw[t], 16);
      else if (p.qmul != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.Kout) m4[e] = p.qmul[n + e];
      }
    }
    if constexpr (kQ8) {
      const floatx4 mq = {m4[0], m4[1], m4[2], m4[3]};
      const int a0 = s.x + b4[0], a1 = s.y + b4[1], a2 = s.z + b4[2], a3 = s.w + b4[3];
      const unsigned w = rbase != nullptr ? requant4<true>(a0, a1, a2, a3, mq, rq, p) : requant4<false>(a0, a1, a2, a3, mq, 0u, p);
      int8_t* y = ybase + (int64_t)m * p.ycs + n;
      if (vec) *reinterpret_cast<unsigned*>(y) = w;
      else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.Kout) y[e] = (int8_t)(w >> (8 * e));
      }
    } else if constexpr (EpiTraits<Epi>::quant) {
      TOut* y = ybase + (int64_t)m * p.ycs + n;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= p.Kout) break;
        const int v = s[e] + b4[e];
        if constexpr (std::is_same<TOut, int>::value) y[e] = v;
        else y[e] = epi_act((float)v * m4[e] + r4[e], p.act, p.act_a, p.act_b);
      }
    } else {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(s[e], p.alpha, b4[e]);
      if (p.res_after_act) epi_act_n<EpiTraits<Epi>::rich>(v, p.act, p.act_a, p.act_b);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += r4[e];
      if (!p.res_after_act) epi_act_n<EpiTraits<Epi>::rich>(v, p.act, p.act_a, p.act_b);
      TOut* y = ybase + y_row_off(p, m) + y_col_off(p, n);
      if (vec) {
        if constexpr (sizeof(TOut) == 4) *reinterpret_cast<floatx4*>(y) = (floatx4){v[0], v[1], v[2], v[3]};
        else *reinterpret_cast<uintx2*>(y) = uintx2{pack2<TOut>(v[0], v[1]), pack2<TOut>(v[2], v[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= p.Kout) break;
          if constexpr (sizeof(TOut) == 4) y[e] = v[e];
          else Store<TOut>::st(y + e, v[e]);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
namespace {

template <typename TIn, typename Epi, int MB, int NB, int NW>
hipError_t launch_tile(const IgemmParams& p, const int epi_vec, SlimArgs a, const int mode, hipStream_t stream) {
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  const int64_t tm = (M + MB * 16 - 1) / (MB * 16), tn = ((int64_t)p.Kout + NB * 16 - 1) / (NB * 16);
  if (tm * tn <= 0 || tm * tn > 0x7fffffff || p.batch > 65535) return hipErrorInvalidValue;
  a.tiles_m = (int)tm;
  a.tiles_n = (int)tn;
  a.t_div = a.m_fast ? a.tiles_m : a.tiles_n;
  div_magic(a.t_div, &a.t_magic, &a.t_shift);
  constexpr size_t lds = (size_t)NW * MB * 16 * (NB * 16 + 4) * 4;
  const dim3 grid((unsigned)(tm * tn), 1, (unsigned)p.batch), block(NW * 64);
  static_assert(lds <= 65536, "more than a launch may ask for by itself");
#define SLIM_LAUNCH(MODE_) hipLaunchKernelGGL((igemm_slim_kernel<TIn, Epi, MB, NB, NW, MODE_>), grid, block, lds, stream, p, epi_vec, a)
  if constexpr (std::is_same<TIn, f16_t>::value || std::is_same<TIn, bf16_t>::value) {
    if (mode == SLIM_LN32) { SLIM_LAUNCH(SLIM_LN32); return hipGetLastError(); }
  }
  if constexpr (sizeof(TIn) > 1) {
    if (mode == SLIM_LN) { SLIM_LAUNCH(SLIM_LN); return hipGetLastError(); }
  }
  if (mode > SLIM_ANY) return hipErrorInvalidValue;
  if (mode == SLIM_ROW) SLIM_LAUNCH(SLIM_ROW);
  else if (mode == SLIM_TAP) SLIM_LAUNCH(SLIM_TAP);
  else SLIM_LAUNCH(SLIM_ANY);
#undef SLIM_LAUNCH
  return hipGetLastError();
}

template <typename TIn, typename Epi>
hipError_t launch_slim(const IgemmParams& p, const int epi_vec, const int variant, hipStream_t stream) {
  constexpr int ES = sizeof(TIn);
  SlimArgs a;
  a.cvec = p.C * ES / 16;
  const int64_t vecs = (int64_t)p.R * p.S * a.cvec;
  if (vecs <= 0 || vecs > (1 << 28)) return hipErrorInvalidValue;
  a.steps = (int)((vecs + 3) / 4);
  div_magic(a.cvec, &a.cv_magic, &a.cv_shift);
  div_magic(p.S, &a.s_magic, &a.s_shift);
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  // one XCD keeps the larger operand's tiles: with fewer pixels than channels the workgroups of one channel tile sit together
  a.m_fast = M < p.Kout;
  const bool row = p.R == 1 && p.S == 1 && p.ph == 0 && p.pw == 0 && (int64_t)(p.Ho - 1) * p.sh < p.H && (int64_t)(p.Wo - 1) * p.sw < p.W;
  const int mode = p.ln ? (p.ln_dt == p.in_dt ? SLIM_LN : SLIM_LN32) : row ? SLIM_ROW : (a.cvec % 4 == 0 ? SLIM_TAP : SLIM_ANY);
  switch (variant) {
    case 1: return launch_tile<TIn, Epi, 1, 1, 16>(p, epi_vec, a, mode, stream);
    case 2: return launch_tile<TIn, Epi, 2, 2, 8>(p, epi_vec, a, mode, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// Which kernel a launch gets, by an estimate of its time in us (beside the launch itself):
//   c0 + c1 * chain + c2 * tiles / 256 + c3 * tiles * stages / 256
// chain: K stages of 128 bytes that one wavefront walks; tiles: of the kernel's own size.  The
// coefficients are a least-squares fit to launches of ResNet-50 at 1 .. 48 images in three types,
// BERT-base at 1 .. 64 sequences and YOLOv3 at 1 .. 16 images, of which each kernel's fit saw those
// where it came within a factor of two of the best (three for the 128 x 128 row, which stands for
// all kernels of igemm.hip and its siblings).  A kernel trace of 2225 such launches, each with
// every kernel that can compute it: estimate + 2.1 us (what a duration holds of the launch itself)
// is off by 8 .. 24 % rms per kernel and type, and the launches as chosen take 2.8 % more than with
// the best kernel for each (16 % in one network: ResNet-50 int8 at one image).  Sums of the
// launches of a step with the wide kernels alone and as chosen: ResNet-50 fp16 at 1 / 4 / 16
// images 0.62 / 0.65 / 0.77 -> 0.28 / 0.38 / 0.63 ms, fp32 at 4 images 2.9 -> 0.72 ms, BERT-base
// fp32 at 2 x 128 tokens 3.7 -> 0.96 ms.  (8-bit coefficients: refitted to the K loop of all requests
// at once.  The 2- and 4-byte ones are older and estimate four of eight kernels 13 .. 19 % too long; refitting them
// too gave 1.2 % over all launches, and BERT-base bf16 at 1 x 41 tokens 389 -> 399 us.)
namespace {
struct SlimCost { float fix, chain, tile, work; };
struct SlimCosts { SlimCost wide, k16, k8, mid; };
constexpr SlimCosts kCost1 = {{4.9f, .37f, 1.4f, .044f}, {0.f, .49f, 2.05f, .045f}, {.66f, 1.04f, .86f, .083f}, {.79f, .25f, 1.49f, .054f}};
constexpr SlimCosts kCost2 = {{4.4f, .42f, 1.0f, .42f}, {.05f, .62f, 2.27f, .056f}, {.73f, .88f, .82f, .108f}, {1.74f, .18f, 1.06f, .16f}};
constexpr SlimCosts kCost4 = {{1.8f, 2.05f, 6.9f, .144f}, {0.f, .59f, 2.07f, .075f}, {1.14f, .93f, 1.15f, .19f}, {2.5f, .344f, 1.78f, .42f}};
// How much faster than the 128 x 128 tiles the choice has to be.  (0.85 .. 1 cost the same over
// all launches.)  2-byte types with more than two 64 x 64 tiles per compute unit: 0.7 - they ask the
// L2s for twice the bytes per operation, which a launch that runs beside this one (the other half of
// a batch) feels: YOLOv3 at 16 images in two halves 2.27 -> 2.34 ms with 0.88 there.  (8-bit layers
// of that size are bound by their results: 1 against 0.7 there takes 427 instead of 449 us for the
// launches of ResNet-50 on 13 images.)
constexpr float kSlimMargin = 0.88f, kSlimMarginFull = 0.7f;
}  // namespace

int igemm_slim_variant(const IgemmParams& p, const bool frag, float* us) {
  if (us != nullptr) *us = 0.f;
  if (p.slim >= 0) return p.slim;
  if (p.f_y != nullptr || p.row_softmax != 0 || p.fixed_order) return 0;
  // what the kernels' addressing assumes: 32-bit offsets inside an image, no column of K behind the packed rows
  // (a tile of 32 pixels touches at most 32 images; weights: 32 rows of the fragment copy, 16 packed ones)
  const int es = dtype_size(p.in_dt);
  if (es == 0 || (int64_t)(p.N < 32 ? p.N : 32) * p.H * p.W * p.xcs * es >= (1ll << 31) || (int64_t)p.R * p.S * p.C > p.w_cols) return 0;
  if ((int64_t)p.w_rs * es >= (1ll << 25)) return 0;
  if (const char* force = getenv("ODLA_HIP_IGEMM_TILE")) {  // tuning aid: "slim1", "slim2", "mid"
    if (strncmp(force, "slim", 4) == 0 && force[4] >= '1' && force[4] <= '2') return force[4] - '0';
    if (strcmp(force, "mid") == 0) return frag ? 3 : 0;
    if (force[0] != 0) return 0;
  }
  // (a tuning aid of another kernel asks for that kernel)
  for (const char* aid : {"ODLA_HIP_WREG_SLICES", "ODLA_HIP_WREG_KSPLIT", "ODLA_HIP_WREG_ROWS", "ODLA_HIP_C3_MIN_FILL", "ODLA_HIP_C3_BC", "ODLA_HIP_C3_SLICES",
                          "ODLA_HIP_LEAN_TILES", "ODLA_HIP_STREAM_WGS"})
    if (getenv(aid) != nullptr) return 0;
  const SlimCosts& c = es == 1 ? kCost1 : es == 2 ? kCost2 : kCost4;
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  const float stages = (float)(((int64_t)p.R * p.S * p.C * es + 127) / 128);
  auto cost = [&](const SlimCost& k, const int tile, const int waves) {
    const float tiles = (float)((M + tile - 1) / tile) * (float)((p.Kout + tile - 1) / tile) * (float)p.batch / 256.f;
    return k.fix + k.chain * stages / (float)waves + k.tile * tiles + k.work * tiles * stages;
  };
  const float t1 = cost(c.k16, 16, 16), t2 = cost(c.k8, 32, 8), t3 = cost(c.mid, 64, 1);
  int v = t1 < t2 ? 1 : 2;
  float t = t1 < t2 ? t1 : t2;
  if (frag && t3 < t) { v = 3; t = t3; }
  if (us != nullptr) *us = t;
  const int64_t tiles64 = ((M + 63) / 64) * (((int64_t)p.Kout + 63) / 64) * p.batch;
  const float margin = v == 3 && es == 2 && tiles64 > 512 ? kSlimMarginFull : kSlimMargin;
  return t < margin * cost(c.wide, 128, 1) ? v : 0;
}

// A product that runs here, of whole rows that the wavefronts of a workgroup can hold.
bool igemm_slim_ln_ok(const IgemmParams& p, const bool frag) {
  if (!p.ln || !dtype_is_float(p.in_dt) || (p.ln_dt != p.in_dt && p.ln_dt != DT_F32)) return false;
  if (p.R != 1 || p.S != 1 || p.sh != 1 || p.sw != 1 || p.ph != 0 || p.pw != 0 || p.Ho != p.H || p.Wo != p.W || p.x_bs != 0) return false;
  const int row = p.C * dtype_size(p.in_dt);
  const int v = igemm_slim_variant(p, frag);
  const int waves = v == 1 ? 16 : v == 2 ? 8 : 0;
  return waves > 0 && row % 64 == 0 && row / 64 >= waves && row / 64 <= kSlimLnSteps * waves;
}

hipError_t launch_igemm_slim(const IgemmParams& p, int epi_vec, int variant, hipStream_t stream) {
  if (variant == 3) return launch_igemm_mid(p, epi_vec, stream);
  const bool rich = p.act == ACT_GELU_ERF || p.act == ACT_GELU_TANH || p.act == ACT_SIGMOID || p.act == ACT_TANH;
  switch (p.in_dt) {
    case DT_F32:
      if (p.out_dt != DT_F32) return hipErrorInvalidValue;
      if (rich) return launch_slim<float, EpiFloat<float, true>>(p, epi_vec, variant, stream);
      return launch_slim<float, EpiFloat<float>>(p, epi_vec, variant, stream);
    case DT_F16:
      if (p.out_dt == DT_F16 && rich) return launch_slim<f16_t, EpiFloat<f16_t, true>>(p, epi_vec, variant, stream);
      if (p.out_dt == DT_F16) return launch_slim<f16_t, EpiFloat<f16_t>>(p, epi_vec, variant, stream);
      if (p.out_dt == DT_F32) return launch_slim<f16_t, EpiFloat<float>>(p, epi_vec, variant, stream);
      return hipErrorInvalidValue;
    case DT_BF16:
      if (p.out_dt == DT_BF16 && rich) return launch_slim<bf16_t, EpiFloat<bf16_t, true>>(p, epi_vec, variant, stream);
      if (p.out_dt == DT_BF16) return launch_slim<bf16_t, EpiFloat<bf16_t>>(p, epi_vec, variant, stream);
      if (p.out_dt == DT_F32) return launch_slim<bf16_t, EpiFloat<float>>(p, epi_vec, variant, stream);
      return hipErrorInvalidValue;
    case DT_I8:
      if (p.out_dt == DT_I8) return p.qmul == nullptr ? hipErrorInvalidValue : launch_slim<int8_t, EpiQuant<0>>(p, epi_vec, variant, stream);
      if (p.out_dt == DT_F32) return p.qmul == nullptr ? hipErrorInvalidValue : launch_slim<int8_t, EpiQuant<1>>(p, 0, variant, stream);
      if (p.out_dt == DT_I32) return launch_slim<int8_t, EpiQuant<2>>(p, 0, variant, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ohip
