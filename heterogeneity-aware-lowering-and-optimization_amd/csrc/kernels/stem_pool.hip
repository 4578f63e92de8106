// The front of a classifier in one launch: a 7 x 7 convolution of stride 2 over a three-channel image,
// ReLU and the 3 x 3 maximum of stride 2 behind it
// [ref: the reference runs the three as operators of their own, ODLA/platforms/dnnl/odla_dnnl.cc].
//
// As launches of their own - the image to its space-to-depth form, the convolution as a 4 x 4 one over that,
// the pool - they cross memory with everything in between: 256 fp16 images of 224 x 224 write and read a
// space-to-depth image of 103 MB and a convolution result of 411 MB for 154 MB in and 103 MB out.
// Here a wavefront takes a strip of pooled rows, 14 pooled columns and all 64 channels (32 for few
// images) of one image:
//   - the source rows are converted to space-to-depth pixels (16 values per 2 x 2 block:
//     (py * 2 + px) * 3 + channel, the order of the packed weights) in a ring of eight rows in LDS; the rows of the
//     next but one step are on their way while a step computes;
//   - the fragment-ordered weights stay in registers and every convolution row is 2 x 16 (8-bit: 2 x 8) matrix
//     instructions on operands straight from LDS, requested three steps ahead (without that: 146 us where this takes 115);
//   - lane l of a half wavefront holds convolution column 14 (l / 16) + l % 16 of 29, so that the three columns of
//     a pooled one sit in one row of 16 lanes.  The maximum over rows is one of registers, the one over columns two
//     lane shifts, on 16-bit results as they are stored, two at a time, or on 8-bit ones' sums: bias, ReLU,
//     rounding and requantisation keep the order of values;
//   - 14 pooled pixels of 64 channels leave as 16-byte vectors, contiguous in a result of its own (one whose only reader is
//     a Concat along the channels is a slice of that one's: its pixels lie a larger pitch apart).
// No barrier: wavefronts drift apart, one in its matrix instructions while the other of its SIMD converts and
// stores (a workgroup of four that filled a patch first and then computed took 251 us).  Bound by both together:
// at 256 fp16 images the matrix cores are busy for 44 % of the time, vector instructions are 72 % of what is issued, and
// 257 MB take 52 us (8 bit: 28 %, 80 %).
// Measured, launches before and now: 256 x 224 x 224 fp16 43 + 203 + 98 us -> 110 - 121 us from card to card, 8 bit
// 38 + 109 + 55 -> 85; one image fp16 4.3 + 8.9 + 4.1 -> 6.8; 13 x 237 x 237 8 bit 7.2 + 16.2 + 5.2 -> 12.3.
// Strips read the rows between them twice, so that a small image in host memory, which the conversion read in place, is
// copied by a launch first: still 2 - 8 us of a call less (one fp16 image into ResNet-50, 96 x 96 280 -> 272 us, 224 x 224
// 336 -> 333, 288 x 288 386 -> 384).
#include "igemm_common.h"

namespace ohip {
namespace {

constexpr int kCols = 14;                                // pooled columns of a wavefront
constexpr int kPatchCols = 2 * kCols + 1 + 3;            // its space-to-depth columns: convolution columns and three more taps
constexpr int kRing = 8;                                 // patch rows held: six that are read (one only where a row outside is replaced), two that are written
static_assert(kPatchCols == 32, "half a wavefront fills a patch row");

// the value of the next lane (within a row of 16; the last one's is not used)
__device__ __forceinline__ int next_lane(const int v) { return __builtin_amdgcn_mov_dpp(v, 0x101, 0xf, 0xf, true); }   // row_shl:1
// largest of two 16-bit values each
__device__ __forceinline__ unsigned max_pairs(const unsigned a, const unsigned b) {
  typedef unsigned short ushortx2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(ushortx2, a), __builtin_bit_cast(ushortx2, b)));
}

// A value as it is stored (8-bit: the level of the quantised value minus 128).  The quotient is that of the division:
// with inv the reciprocal rounded to nearest, one step on the remainder, which the fma has exactly, gives the quotient
// rounded to nearest [Markstein, Computation of elementary functions on the IBM RISC System/6000 processor, 1990].
// What is far outside the levels is cut first, with infinities (a NaN is the lowest level, as the division's is).
struct StemLevels { float scale, inv, most; int zp; };
template <typename T>
__device__ __forceinline__ unsigned stem_bits(const float v, const StemLevels&) {
  T t;
  Store<T>::st(&t, v);
  return t.bits;
}
template <>
__device__ __forceinline__ unsigned stem_bits<int8_t>(const float v, const StemLevels& l) {
  const float c = __builtin_amdgcn_fmed3f(v, -l.most, l.most), q = c * l.inv;
  float t = rintf(__builtin_fmaf(__builtin_fmaf(-q, l.scale, c), l.inv, q)) + (float)l.zp;
  t = fminf(fmaxf(t, 0.f), 255.f);
  return (unsigned)(uint8_t)q_to_stored((int)t);
}
constexpr float kScaleLeast = 0x1p-80f, kScaleMost = 0x1p+80f;     // nothing above leaves the range of normal numbers

// the six pairs of source pixels behind one space-to-depth pixel, as they were read
struct StemRaw { float v[2][3][2]; };

template <typename T, int NJ>   // NJ: 32-channel blocks of a wavefront
__global__ void __launch_bounds__(64, 2) stem_pool_kernel(const StemPoolParams p, const StemLevels levels, const int rows) {
  using Acc = typename Mma<T>::Acc;
  constexpr int ES = sizeof(T), PX = 16 * ES;            // bytes of a space-to-depth pixel
  constexpr int NKK = 16 * PX / 32;                      // 32-byte K steps of the 16 taps
  constexpr int PITCH = kPatchCols * PX;                 // bytes of a patch row
  constexpr int OPITCH = NJ * 32 * ES + 16;                   // bytes of a staged result pixel
  __shared__ __attribute__((aligned(16))) unsigned char patch[kRing * PITCH];
  __shared__ __attribute__((aligned(16))) unsigned char stage[kCols * OPITCH];
  __shared__ __attribute__((aligned(16))) unsigned s_bias[64], s_mul[64];

  const int lane = threadIdx.x, l32 = lane & 31, lg = lane >> 5, l16 = lane & 15;
  // neighbouring strips share source rows: one XCD (workgroups are dealt round-robin)
  int bid = blockIdx.x;
  {
    const int per = gridDim.x >> 3;
    if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
  }
  const int c0 = NJ == 1 ? (bid & 1) * 32 : 0;                     // the first channel
  if (NJ == 1) bid >>= 1;
  const int strips = (p.Po + rows - 1) / rows, col_groups = (p.Qo + kCols - 1) / kCols;
  const int cg = bid % col_groups, t_ = bid / col_groups, n = t_ / strips, p0 = (t_ - n * strips) * rows;
  const int count = rows < p.Po - p0 ? rows : p.Po - p0;           // pooled rows of this strip
  const int q0 = cg * kCols;                                       // its first pooled column
  const int ho0 = 2 * p0 - 1, wo0 = 2 * q0 - 1;                    // the first convolution row and column

  // ---- the patch: pixel (row, col) is the space-to-depth image's (ho0 - ph + row, wo0 - pw + col); lane l requests
  // column l % 32 of rows l / 32 and beyond, always at a position inside the image, and it is replaced where that
  // is another one ----
  const int64_t plane = (int64_t)p.H * p.W;
  const float* img = p.x + (int64_t)n * 3 * plane;
  const bool pairs = (p.W & 1) == 0 && (reinterpret_cast<uintptr_t>(p.x) & 7u) == 0;
  const int x0 = 2 * (wo0 - p.pw + l32), h0 = 2 * (ho0 - p.ph + lg);
  auto request = [&](const int row, StemRaw& raw) __attribute__((always_inline)) {
#pragma unroll
    for (int py = 0; py < 2; ++py) {
      const int h = h0 + 2 * row + py;
      const unsigned line = (unsigned)(h < 0 ? 0 : h < p.H ? h : p.H - 1) * (unsigned)p.W;
      if (pairs) {
        typedef float floatx2 __attribute__((ext_vector_type(2)));
        const unsigned at = line + (unsigned)(x0 < 0 ? 0 : x0 < p.W ? x0 : p.W - 2);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const floatx2 v = *reinterpret_cast<const floatx2*>(img + c * plane + at);
          raw.v[py][c][0] = v.x;
          raw.v[py][c][1] = v.y;
        }
      } else {
#pragma unroll
        for (int px = 0; px < 2; ++px) {
          const unsigned at = line + (unsigned)(x0 + px < 0 ? 0 : x0 + px < p.W ? x0 + px : p.W - 1);
#pragma unroll
          for (int c = 0; c < 3; ++c) raw.v[py][c][px] = (img + c * plane)[at];
        }
      }
    }
  };
  const bool in0 = x0 >= 0 && x0 < p.W, in1 = x0 + 1 >= 0 && x0 + 1 < p.W;
  auto keep = [&](const int row, const StemRaw& raw) __attribute__((always_inline)) {
    const int h = h0 + 2 * row;
    const bool ok[2][2] = {{in0 && h >= 0 && h < p.H, in1 && h >= 0 && h < p.H}, {in0 && h + 1 >= 0 && h + 1 < p.H, in1 && h + 1 >= 0 && h + 1 < p.H}};
    constexpr int PW = 4 / ES;
    unsigned word[16 / PW];
#pragma unroll
    for (int q = 0; q < 16 / PW; ++q) {
      word[q] = 0u;
#pragma unroll
      for (int e = 0; e < PW; ++e) {
        const int c = q * PW + e, py = (c / 3) >> 1, px = (c / 3) & 1;   // (behind the twelfth: values that meet zero weights)
        if (c < 12) word[q] |= stem_bits<T>(ok[py][px] ? raw.v[py][c % 3][px] : 0.f, levels) << (e * 8 * ES);
      }
    }
    uintx4* dst = reinterpret_cast<uintx4*>(patch + ((row + lg) & (kRing - 1)) * PITCH + l32 * PX);
#pragma unroll
    for (int q = 0; q < PX / 16; ++q) dst[q] = uintx4{word[q * 4], word[q * 4 + 1], word[q * 4 + 2], word[q * 4 + 3]};
  };
  // a wavefront is a workgroup and its LDS operations complete in issue order
  auto ordered = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // ---- everything the first pooled row needs is requested at once ----
  StemRaw first[3], ahead;
#pragma unroll
  for (int i = 0; i < 3; ++i) request(2 * i, first[i]);
  uintx4 w[NJ][NKK];
  {
    const uintx4* wf = reinterpret_cast<const uintx4*>(p.w_frag) + (c0 / 32) * p.wf_chunks * 64 + lane;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) w[j][kk] = wf[(j * p.wf_chunks + kk) * 64];
  }
  s_bias[lane] = p.bias != nullptr ? reinterpret_cast<const unsigned*>(p.bias)[lane] : 0u;
  s_mul[lane] = p.qmul != nullptr ? reinterpret_cast<const unsigned*>(p.qmul)[lane] : 0u;
#pragma unroll
  for (int i = 0; i < 3; ++i) keep(2 * i, first[i]);
  if (count > 1) request(6, ahead);
  ordered();

  // this lane's convolution column behind wo0 (lane 15 of a row of 16 is not used; a column outside the result is
  // replaced by its neighbour, which is in the same window)
  const int wlast = p.Wo - 1 - wo0, hlast = p.Ho - 1 - ho0;
  int lcol = l32 == 31 ? 2 * kCols : (l32 >> 4) * kCols + l16;
  lcol = wo0 + lcol < 0 ? 1 : lcol < wlast ? lcol : wlast;
  // K step kk: 2-byte operands one tap, its halves for the two lane groups; 8-bit ones two taps
  const unsigned char* a0 = patch + lcol * PX + lg * 16;

  // what is held of a convolution row: 16-bit results as they are stored, in pairs; 8-bit ones' sums
  constexpr int NH = ES == 1 ? 4 : 2;
  typedef unsigned Held[NJ][4][NH];
  auto row_of = [&](const int r, Held& held) __attribute__((always_inline)) {
    Acc acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = 0;
    auto operand = [&](const int kk) __attribute__((always_inline)) {
      constexpr int KPT = NKK / 4;                       // K steps of a filter row
      return *reinterpret_cast<const uintx4*>(a0 + ((r + kk / KPT) & (kRing - 1)) * PITCH + (kk % KPT) * 32);
    };
    // requested three steps before they are multiplied
    constexpr int kAhead = 3;
    uintx4 v[kAhead + 1];
#pragma unroll
    for (int kk = 0; kk < kAhead; ++kk) v[kk] = operand(kk);
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      if (kk + kAhead < NKK) v[(kk + kAhead) % (kAhead + 1)] = operand(kk + kAhead);
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[j] = Mma<T>::run(w[j][kk], v[kk % (kAhead + 1)], acc[j]);
      if (kk + kAhead < NKK) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, NJ, 0);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if constexpr (ES == 1) {
#pragma unroll
          for (int e = 0; e < 4; ++e) held[j][q][e] = (unsigned)acc[j][q * 4 + e];
        } else {
          const floatx4 b = *reinterpret_cast<const floatx4*>(s_bias + c0 + j * 32 + q * 8 + lg * 4);
          float f[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f[e] = acc[j][q * 4 + e] + b[e];
            f[e] = f[e] > 0.f ? f[e] : 0.f;
          }
          held[j][q][0] = pack2<T>(f[0], f[1]);
          held[j][q][1] = pack2<T>(f[2], f[3]);
        }
  };
  // (what ReLU leaves orders as the whole numbers of its bits; requantisation keeps the order of the sums)
  auto larger = [&](const unsigned a, const unsigned b) __attribute__((always_inline)) {
    if constexpr (ES == 1) return (unsigned)((int)a > (int)b ? (int)a : (int)b);
    else return max_pairs(a, b);
  };
  auto finish = [&](const int prow, const Held& best) __attribute__((always_inline)) {
    const bool mine = (l16 & 1) == 0 && l16 < kCols;
    unsigned char* out = stage + ((l32 >> 4) * (kCols / 2) + (l16 >> 1)) * OPITCH + lg * 4 * ES;
    unsigned m[NJ][4][NH];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int e = 0; e < NH; ++e) {
          m[j][q][e] = larger(best[j][q][e], (unsigned)next_lane((int)best[j][q][e]));
          m[j][q][e] = larger(m[j][q][e], (unsigned)next_lane((int)m[j][q][e]));
        }
        if constexpr (ES == 1) {
          const int ch = c0 + j * 32 + q * 8 + lg * 4;
          const intx4 b = *reinterpret_cast<const intx4*>(s_bias + ch);
          const floatx4 mul = *reinterpret_cast<const floatx4*>(s_mul + ch);
          IgemmParams qp;
          qp.q_add = p.q_add;
          qp.q_lo = p.q_lo;
          m[j][q][0] = requant4<false>((int)m[j][q][0] + b.x, (int)m[j][q][1] + b.y, (int)m[j][q][2] + b.z, (int)m[j][q][3] + b.w, mul, 0u, qp);
        }
      }
    if (mine) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if constexpr (ES == 1) *reinterpret_cast<unsigned*>(out + j * 32 + q * 8) = m[j][q][0];
          else *reinterpret_cast<uintx2*>(out + (j * 32 + q * 8) * 2) = uintx2{m[j][q][0], m[j][q][1]};
    }
    ordered();
    T* y = reinterpret_cast<T*>(p.y) + (((int64_t)n * p.Po + prow) * p.Qo + q0) * p.ycs + c0;
    constexpr int CH = NJ * 32 * ES / 16;                // 16-byte pieces of a pixel
#pragma unroll
    for (int k = 0; k < (kCols * CH + 63) / 64; ++k) {
      const int piece = k * 64 + lane, px = piece / CH, c = piece % CH;
      if (piece < kCols * CH && q0 + px < p.Qo)
        *reinterpret_cast<uintx4*>(reinterpret_cast<unsigned char*>(y) + px * p.ycs * ES + c * 16) = *reinterpret_cast<const uintx4*>(stage + px * OPITCH + c * 16);
    }
    ordered();
  };

  // convolution rows 2 k, 2 k + 1 and 2 k + 2 of the strip are pooled row k; the last one is also the next one's
  // first.  One outside the result is replaced by its neighbour, which is in the same window.
  Held best;
  row_of(ho0 < 0 ? 1 : 0, best);
#pragma unroll 1
  for (int k = 0; k < count; ++k) {
    // patch rows 2 k to 2 k + 5 are read in this step; the two the next one reads besides replace 2 k - 2 and
    // 2 k - 1, and the two behind those are on their way while this step computes
    if (k + 1 < count) {
      keep(2 * k + 6, ahead);
      if (k + 2 < count) request(2 * k + 8, ahead);
      ordered();
    }
    Held next;
    row_of(2 * k + 1 < hlast ? 2 * k + 1 : hlast, next);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < NH; ++e) best[j][q][e] = larger(best[j][q][e], next[j][q][e]);
    row_of(2 * k + 2 < hlast ? 2 * k + 2 : hlast, next);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < NH; ++e) best[j][q][e] = larger(best[j][q][e], next[j][q][e]);
    finish(p0 + k, best);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < NH; ++e) best[j][q][e] = next[j][q][e];
  }
}

// Up to so many wavefronts each takes one 32-channel block instead of both (the slots of the chip are free): one fp16
// image 6.8 us for 8.1, two 7.9 for 8.8, four 8.3 for 9.4, four 8-bit ones 8.4 for 8.7.
constexpr int64_t kHalves = 2048;
// Pooled rows of a strip: two wavefronts of each SIMD at a time, and a strip costs about two rows more than it has (the
// requests of its first row, its first convolution row).  The number of strips with the least of (rounds of
// wavefronts) x (rows of a strip + 2).  256 fp16 images: strips of 28 rows in one round 121 us, of 14 in two 125, of
// 56 with one wavefront a SIMD 195; 13 8-bit ones of 60 rows: 2 rows a strip in one round 12.3 us, 1 row 14.8, 4 rows 15.6.
int strip_rows(const StemPoolParams& p) {
  constexpr int64_t kSlots = 2048;
  const int64_t columns = (int64_t)p.N * ((p.Qo + kCols - 1) / kCols);
  int rows = p.Po;
  int64_t least = INT64_MAX;
  for (int strips = 1; strips <= p.Po && strips <= 256; ++strips) {
    const int r = (p.Po + strips - 1) / strips;
    const int64_t waves = columns * ((p.Po + r - 1) / r), cost = ((waves + kSlots - 1) / kSlots) * (r + 2);
    if (cost < least) least = cost, rows = r;
  }
  return rows;
}

template <typename T>
hipError_t launch_rows(const StemPoolParams& p, hipStream_t stream) {
  const int rows = strip_rows(p);
  const int64_t grid = (int64_t)p.N * ((p.Po + rows - 1) / rows) * ((p.Qo + kCols - 1) / kCols);
  if (grid > 0x3fffffff) return hipErrorInvalidValue;
  const StemLevels levels{p.scale, 1.f / p.scale, 1024.f * p.scale, p.zp};
  if (2 * grid <= kHalves) hipLaunchKernelGGL((stem_pool_kernel<T, 1>), dim3((unsigned)(2 * grid)), dim3(64), 0, stream, p, levels, rows);
  else hipLaunchKernelGGL((stem_pool_kernel<T, 2>), dim3((unsigned)grid), dim3(64), 0, stream, p, levels, rows);
  return hipGetLastError();
}

}  // namespace

bool stem_pool_supported(const StemPoolParams& p) {
  if (p.dt != DT_F16 && p.dt != DT_BF16 && p.dt != DT_I8) return false;
  if (p.N <= 0 || p.H < 2 || p.W < 2 || p.Ho <= 0 || p.Wo <= 0 || p.Po <= 0 || p.Qo <= 0) return false;
  if (p.dt == DT_I8 && !(p.scale >= kScaleLeast && p.scale <= kScaleMost)) return false;
  // whole 16-byte vectors of a result pixel
  if (p.ycs < 64 || p.ycs > (1 << 24) || p.ycs % (16 / dtype_size(p.dt)) != 0) return false;
  // every pooled value covers a convolution value; source coordinates and one image's elements in 32 bits
  if (2 * ((int64_t)p.Po - 1) - 1 >= p.Ho || 2 * ((int64_t)p.Qo - 1) - 1 >= p.Wo) return false;
  return (int64_t)p.H * p.W < (1ll << 29) && p.ph >= 0 && p.ph < 4 && p.pw >= 0 && p.pw < 4;
}

hipError_t launch_stem_pool(const StemPoolParams& p, hipStream_t stream) {
  if (!stem_pool_supported(p) || p.x == nullptr || p.y == nullptr || p.w_frag == nullptr || p.wf_chunks < (p.dt == DT_I8 ? 8 : 16)) return hipErrorInvalidValue;
  if (((reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.w_frag)) & 15u) != 0 || (p.dt == DT_I8 && p.qmul == nullptr)) return hipErrorInvalidValue;
  switch (p.dt) {
    case DT_F16: return launch_rows<f16_t>(p, stream);
    case DT_BF16: return launch_rows<bf16_t>(p, stream);
    default: return launch_rows<int8_t>(p, stream);
  }
}

}  // namespace ohip
