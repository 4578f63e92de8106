// Implicit GEMM on 64 pixel x 64 channel tiles with both operands loaded straight into LDS:
// launches whose 128 x 128 tiles would leave compute units idle, but which have too much work
// for the direct operand loads of igemm_slim.hip.
//
// Four wavefronts own the quadrants of a tile (one 32x32 MFMA block each); a K stage is 128
// bytes of 64 pixel rows and of 64 weight rows (16 KiB), brought in by direct-to-LDS loads into a
// ring of four, three stages ahead.  Per stage a wavefront issues four requests and eight
// fragment reads for four MFMA steps; fragments are read one stage ahead of their MFMAs, so that
// neither the request nor the LDS latency is on the chain.
// (Measured and left out: two K groups of four wavefronts with a ring each; eight wavefronts that
//  take half of every stage each, 3x3 256 -> 256 on 13 maps of 15 x 15 8.8 -> 8.7 us and 1x1 layers 4 %
//  slower; a ring of eight, which only long runs of K over 1x1 filters gain from.)
// A launch here is 4 - 12 us, of which the K loop is a third to two thirds (clock stamps): what the
// epilogue needs is requested before the K loop, its arithmetic runs where the accumulators are, and
// the arguments are fetched together.  With the shared epilogue behind the loop (bias, multipliers
// and residual one round trip after the other, results through LDS) and arguments loaded where they
// are named, 8-bit layers of 13 images took: 3x3 256 -> 256 at 15 x 15 9.9 us, 8.8 now; 1x1
// 256 -> 1024 with a residual 12 us, 8.9 now; ResNet-50 int8 on 13 images of 237 x 237 532 -> 502 us.
#include "igemm_common.h"

#include <cstdlib>
#include <cstring>

namespace ohip {

struct MidArgs {
  int tiles_m = 0, tiles_n = 0;
  int m_fast = 0;        // neighbouring workgroups share channels (1) or pixels (0)
  int t_div = 1, t_shift = 0;   // division of a workgroup's number by the tiles of the fast direction
  unsigned t_magic = 0;
  int stages = 0;        // 128-byte K stages
  int cvec = 1;          // 16-byte vectors per tap
  unsigned cv_magic = 0, s_magic = 0;
  int cv_shift = 0, s_shift = 0;
};

// How K maps to taps: one contiguous run per pixel (1x1 filters without padding) / a stage inside
// one tap / any.  In the first two the walk over K is wavefront-uniform (scalar registers); with
// one wavefront per SIMD a stage lasts as long as its instructions, so every one of them counts.
enum MidMode { MID_ROW = 0, MID_TAP = 1, MID_ANY = 2 };

template <typename TIn, typename Epi, int MODE>
__global__ void __launch_bounds__(256, 2)
igemm_mid_kernel(const IgemmParams p, const int epi_vec, const MidArgs a) {
  constexpr int BM = 64, BN = 64, ES = sizeof(TIn);
  constexpr int NBUF = 4, BUF = 16384;
  using Acc = typename Mma<TIn>::Acc;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];   // NBUF * BUF
  fetch_args(p.x, p.w_frag, p.wf_chunks, p.wf_tiles, p.N, p.H, p.W, p.xcs, p.Ho, p.Wo, p.R, p.S, p.sh, p.sw, p.ph, p.pw, p.dh, p.dw, p.howo_magic,
             p.howo_shift, p.wo_magic, p.wo_shift, p.x_bs, p.batch, a.tiles_m, a.tiles_n, a.m_fast, a.t_div, a.t_magic, a.t_shift, a.stages, a.cvec);
  fetch_args(p.bias, p.residual, p.y, p.ycs, p.rcs, p.y_bs, p.r_bs, p.bias_bs, p.y_rdiv, p.y_zdiv, p.alpha, p.act, p.act_a, p.act_b, p.Kout, p.qmul, epi_vec);
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (EpiTraits<Epi>::quant) { WARM_ARG(p, q_add); WARM_ARG(p, r_add); }
#endif

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lg = lane >> 5;
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
  const unsigned char* x = reinterpret_cast<const unsigned char*>(reinterpret_cast<const TIn*>(p.x) + (int64_t)z * p.x_bs);

  // ---- requests of this wavefront: pixel rows wave * 16 + i * 8 + lane / 8 and two weight fragments ----
  const unsigned char* wbase;   // wavefront-uniform
  {
    int t = tile_n * 2 + (wave >> 1);
    t = t < p.wf_tiles ? t : p.wf_tiles - 1;   // surplus channels are computed and never stored
    wbase = reinterpret_cast<const unsigned char*>(p.w_frag) +
            (((int64_t)z * p.wf_tiles + t) * p.wf_chunks + (wave & 1) * 2) * 1024;
  }
  const unsigned lane16 = (unsigned)lane * 16u;
  const uint64_t fill_u = reinterpret_cast<uint64_t>(p.w_frag) + (uint64_t)((int64_t)p.batch * p.wf_tiles * p.wf_chunks * 1024);
  uint64_t a_ptr[2];
  unsigned a_off[2], a_mask[2];
  int a_hi[2], a_wi[2], a_kv[2];
  const int HoWo = p.Ho * p.Wo;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = wave * 16 + i * 8 + (lane >> 3);
    const int m = tile_m * BM + row;
    const bool ok = m < M;
    const int mm = ok ? m : M - 1;                  // surplus rows are computed and never stored
    const int n_img = fast_div(mm, p.howo_magic, p.howo_shift);
    const int rem = mm - n_img * HoWo;
    const int ho = fast_div(rem, p.wo_magic, p.wo_shift);
    const int wo = rem - ho * p.Wo;
    a_hi[i] = ho * p.sh - p.ph;
    a_wi[i] = wo * p.sw - p.pw;
    a_kv[i] = (lane & 7) ^ ((row >> 1) & 7);        // the chunk that belongs in this lane's slot
    const int64_t off = (((int64_t)n_img * p.H + a_hi[i]) * p.W + a_wi[i]) * p.xcs * ES + (MODE == MID_ANY ? 0 : a_kv[i] * 16);
    a_ptr[i] = reinterpret_cast<uint64_t>(x) + (uint64_t)off;
    a_off[i] = (unsigned)off;
    a_mask[i] = 0u;
    if constexpr (MODE == MID_TAP) {                // one validity bit per tap
      unsigned cols = 0u;                           // ... of one filter row, then where the rows are inside
      for (int q = 0; q < p.S; ++q) cols |= (unsigned)((unsigned)(a_wi[i] + q * p.dw) < (unsigned)p.W) << q;
      for (int r = 0; r < p.R; ++r) a_mask[i] |= (unsigned)(a_hi[i] + r * p.dh) < (unsigned)p.H ? cols << (r * p.S) : 0u;
    }
  }
  const int kvecs = p.R * p.S * a.cvec;
  // the uniform walk: bytes left in the tap, tap column, byte offset from tap (0, 0) channel 0, bit of the tap
  const int tap_bytes = a.cvec * 16;
  int left = tap_bytes, ks = 0, toff = 0;
  unsigned tapbit = 1u;
  const int step_s = p.dw * p.xcs * ES - tap_bytes;                                  // behind the last byte of a tap, to the next one
  const int step_r = (p.dh * p.W - (p.S - 1) * p.dw) * p.xcs * ES - tap_bytes;       // ... to the first one of the next filter row
  using lds_ptr = __attribute__((address_space(3))) void*;
  int next = 0;                        // next stage to request
  unsigned char* const dst0 = smem + wave * 2048;
  // (requests behind the last stage repeat it, to keep the count of operations constant)
  auto request = [&](auto buf, auto piece) __attribute__((always_inline)) {
    constexpr int i = decltype(piece)::value;
    unsigned char* dst = dst0 + decltype(buf)::value * BUF + (i & 1) * 1024;
#if defined(__HIP_DEVICE_COMPILE__)  // (the builtin is unknown to the host pass, which only needs the launch stub)
    if constexpr (i >= 2) {
      __builtin_amdgcn_global_load_lds(wbase + (i & 1) * 1024 + lane16, (lds_ptr)(dst + 8192), 16, 0, 0);
    } else if constexpr (MODE == MID_ROW) {
      __builtin_amdgcn_global_load_lds(x + toff + (uint64_t)a_off[i], (lds_ptr)dst, 16, 0, 0);
    } else {
      uint64_t src;
      if constexpr (MODE == MID_TAP) {
        src = (a_mask[i] & tapbit) != 0u ? a_ptr[i] + (int64_t)toff : fill_u;
      } else {
        const int kv = next * 8 + a_kv[i];
        const int tap = fast_div(kv, a.cv_magic, a.cv_shift);
        const int r = fast_div(tap, a.s_magic, a.s_shift);
        const int hoff = r * p.dh, woff = (tap - r * p.S) * p.dw;
        const int off = (hoff * p.W + woff) * p.xcs * ES + (kv - tap * a.cvec) * 16;
        const bool ok = kv < kvecs && (unsigned)(a_hi[i] + hoff) < (unsigned)p.H && (unsigned)(a_wi[i] + woff) < (unsigned)p.W;
        src = ok ? a_ptr[i] + (int64_t)off : fill_u;
      }
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned char*>(src), (lds_ptr)dst, 16, 0, 0);
    }
#else
    (void)dst;
#endif
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (next + 1 < a.stages) {
      ++next;
      wbase += 4096;
      toff += 128;
      if constexpr (MODE == MID_TAP) {
        left -= 128;
        if (left == 0) {
          left = tap_bytes;
          tapbit <<= 1;
          if (++ks == p.S) { ks = 0; toff += step_r; } else toff += step_s;
        }
      }
    }
  };

  Acc acc[1][1];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][0][e] = 0;
  const int wm = wave & 1, wn = wave >> 1;
  // the epilogue's operands: older than every request the K loop counts, so nothing waits for them
  BlockOperands<TIn, Epi> epi;
  BlockResult<TIn, Epi> block;
  epi.fetch(p, epi_vec, z, tile_n * BN + wn * 32, lg);
  block.fetch(p, epi, tile_m * BM + wm * 32 + l32, M);

  // fragments: row l32 of the quadrant, chunk 2 * kk + lg in its swizzled slot; weights lane-major
  const int sw = (l32 >> 1) & 7;
  const unsigned char* rda[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    rda[kk] = smem + (wm * 32 + l32) * 128 + ((lg ^ (sw & 1)) * 16) + (kk ^ (sw >> 1)) * 32;
  const unsigned char* rdw = smem + 8192 + wn * 4096 + lane * 16;
  auto frags = [&](auto buf, uintx4 (&fa)[4], uintx4 (&fw)[4]) __attribute__((always_inline)) {
    constexpr int off = decltype(buf)::value * BUF;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      fa[kk] = *reinterpret_cast<const uintx4*>(rda[kk] + off);
      fw[kk] = *reinterpret_cast<const uintx4*>(rdw + off + kk * 1024);
    }
  };
  // a barrier for direct-to-LDS data: mine has landed (the count), then everyone's has
  auto arrive = [&](auto in_flight) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    constexpr int n = decltype(in_flight)::value;
    __builtin_amdgcn_s_waitcnt(0x0f70 | (n & 15) | (n >> 4) << 14);   // vmcnt only
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  static_for<NBUF - 1>([&](auto b) __attribute__((always_inline)) {
    static_for<4>([&](auto i) __attribute__((always_inline)) { request(b, i); });
    advance();
  });
  arrive(std::integral_constant<int, 4 * (NBUF - 2)>{});
  uintx4 fa[2][4], fw[2][4];
  frags(std::integral_constant<int, 0>{}, fa[0], fw[0]);
  // Stage kt (ring position s): stage kt + 1 has landed for everyone, and everyone's fragments of
  // stage kt - 1 are in registers (their MFMAs came before the barrier), so its buffer takes stage
  // kt + NBUF - 1.  The fragments of kt + 1 are requested behind the MFMAs of kt (ahead of them,
  // the compiler would wait for them too: it does not count LDS reads across the loop's back
  // edge) and travel while the last of these runs and the wavefronts meet at the next barrier.
  for (int kt = 0; kt < a.stages; kt += NBUF) {
    static_for<NBUF>([&](auto s) __attribute__((always_inline)) {
      constexpr int b = decltype(s)::value;
      if (b > 0 && kt + b >= a.stages) return;   // (wavefront-uniform)
      arrive(std::integral_constant<int, 4 * (NBUF - 3)>{});
      // a request behind each MFMA: it is issued while the matrix core works
      static_for<4>([&](auto i) __attribute__((always_inline)) {
        constexpr int kk = decltype(i)::value;
        acc[0][0] = Mma<TIn>::run(fw[b & 1][kk], fa[b & 1][kk], acc[0][0]);
        __builtin_amdgcn_sched_barrier(0);
        request(std::integral_constant<int, (b + NBUF - 1) % NBUF>{}, i);
        __builtin_amdgcn_sched_barrier(0);
      });
      advance();
      frags(std::integral_constant<int, (b + 1) % NBUF>{}, fa[(b + 1) & 1], fw[(b + 1) & 1]);
    });
  }
  // (no request may be in flight when the workgroup ends: its LDS is another's then)
  arrive(std::integral_constant<int, 0>{});
  block.finish(p, epi, acc[0][0]);
}

// ---------------------------------------------------------------------------
namespace {

template <typename TIn, typename Epi>
hipError_t launch_mid(const IgemmParams& p, const int epi_vec, hipStream_t stream) {
  constexpr int ES = sizeof(TIn);
  MidArgs a;
  a.cvec = p.C * ES / 16;
  const int64_t vecs = (int64_t)p.R * p.S * a.cvec;
  if (vecs <= 0 || vecs > (1 << 28)) return hipErrorInvalidValue;
  a.stages = (int)((vecs + 7) / 8);
  if (p.w_frag == nullptr || p.wf_chunks != a.stages * 4) return hipErrorInvalidValue;
  div_magic(a.cvec, &a.cv_magic, &a.cv_shift);
  div_magic(p.S, &a.s_magic, &a.s_shift);
  const int64_t M = (int64_t)p.N * p.Ho * p.Wo;
  const int64_t tm = (M + 63) / 64, tn = ((int64_t)p.Kout + 63) / 64;
  if (tm * tn <= 0 || tm * tn > 0x7fffffff || p.batch > 65535) return hipErrorInvalidValue;
  a.tiles_m = (int)tm;
  a.tiles_n = (int)tn;
  // one XCD keeps the larger operand's tiles
  a.m_fast = M < p.Kout;
  a.t_div = a.m_fast ? a.tiles_m : a.tiles_n;
  div_magic(a.t_div, &a.t_magic, &a.t_shift);
  const dim3 grid((unsigned)(tm * tn), 1, (unsigned)p.batch);
  const bool row = p.R == 1 && p.S == 1 && p.ph == 0 && p.pw == 0 && (int64_t)(p.Ho - 1) * p.sh < p.H && (int64_t)(p.Wo - 1) * p.sw < p.W;
  // (the row form keeps 32-bit byte offsets from the start of the problem's pixels)
  const bool near = (int64_t)p.N * p.H * p.W * p.xcs * ES < (1ll << 31);
  const int mode = a.cvec % 8 != 0 || p.R * p.S > 32 ? MID_ANY : (row && near ? MID_ROW : MID_TAP);
  if (mode == MID_ROW) hipLaunchKernelGGL((igemm_mid_kernel<TIn, Epi, MID_ROW>), grid, dim3(256), 65536, stream, p, epi_vec, a);
  else if (mode == MID_TAP) hipLaunchKernelGGL((igemm_mid_kernel<TIn, Epi, MID_TAP>), grid, dim3(256), 65536, stream, p, epi_vec, a);
  else hipLaunchKernelGGL((igemm_mid_kernel<TIn, Epi, MID_ANY>), grid, dim3(256), 65536, stream, p, epi_vec, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_igemm_mid(const IgemmParams& p, int epi_vec, hipStream_t stream) {
  const bool rich = p.act == ACT_GELU_ERF || p.act == ACT_GELU_TANH || p.act == ACT_SIGMOID || p.act == ACT_TANH;
  switch (p.in_dt) {
    case DT_F32:
      if (p.out_dt != DT_F32) return hipErrorInvalidValue;
      if (rich) return launch_mid<float, EpiFloat<float, true>>(p, epi_vec, stream);
      return launch_mid<float, EpiFloat<float>>(p, epi_vec, stream);
    case DT_F16:
      if (p.out_dt == DT_F16 && rich) return launch_mid<f16_t, EpiFloat<f16_t, true>>(p, epi_vec, stream);
      if (p.out_dt == DT_F16) return launch_mid<f16_t, EpiFloat<f16_t>>(p, epi_vec, stream);
      if (p.out_dt == DT_F32) return launch_mid<f16_t, EpiFloat<float>>(p, epi_vec, stream);
      return hipErrorInvalidValue;
    case DT_BF16:
      if (p.out_dt == DT_BF16 && rich) return launch_mid<bf16_t, EpiFloat<bf16_t, true>>(p, epi_vec, stream);
      if (p.out_dt == DT_BF16) return launch_mid<bf16_t, EpiFloat<bf16_t>>(p, epi_vec, stream);
      if (p.out_dt == DT_F32) return launch_mid<bf16_t, EpiFloat<float>>(p, epi_vec, stream);
      return hipErrorInvalidValue;
    case DT_I8:
      if (p.out_dt == DT_I8) return p.qmul == nullptr ? hipErrorInvalidValue : launch_mid<int8_t, EpiQuant<0>>(p, epi_vec, stream);
      if (p.out_dt == DT_F32) return p.qmul == nullptr ? hipErrorInvalidValue : launch_mid<int8_t, EpiQuant<1>>(p, 0, stream);
      if (p.out_dt == DT_I32) return launch_mid<int8_t, EpiQuant<2>>(p, 0, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ohip
