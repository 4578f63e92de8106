// One-launch attention on gfx950:
//
//   out[b, h] = softmax(scale * q[b, h] . k[b, h]^T + mask[b]) . v[b, h]
//
// for 16-bit operands (bf16 / fp16) and head size 64 - the block that an encoder layer otherwise
// runs as matrix product, Softmax, transposition of v and matrix product, each with its own pass
// over a [B, heads, S, S] tensor
// [ref: the reference compiler matches the same block as one instruction,
//  lib/transforms/fusion.cc:315-348].
//
// One workgroup per (batch, head) and 128 queries, one wavefront per 32 queries.  Up to 128 keys
// are one tile; longer sequences walk tiles of 128 keys with a running maximum and sum per query
// (the next tile's rows travel in registers while the current one is used).  k goes through LDS
// once (rows padded to 144 bytes), v is transposed on its way into LDS, q comes straight from
// global memory into MFMA operand registers.  A launch of few workgroups is a chain of tiles with
// one wavefront per SIMD: there two groups of four wavefronts take every other tile each, and the
// second group's maxima, sums and contexts join the first's through LDS (a chip that is full
// loses: 16 x 512 tokens 30 -> 37 us, 8 x 384 15.4 -> 19.9).
// BERT-base in accuracy mode at 8 x 384 tokens: product, Softmax, transposition and product took
// 22 + 20 + 7 + 14 us per layer, this launch 15.3; at 1 x 41 tokens (keys that fill no block) nine
// launches became one.  With v^T stored value by value, the library's exponential and one group
// throughout / now, us a launch: 8 x 384 18.2 / 15.3, 64 x 128 13.8 / 12.7, 16 x 512 36.6 / 30.7,
// 1 x 512 15.3 / 10.9, 1 x 41 4.2 / 3.9.
//   scores  C[key][query] = k . q^T  (v_mfma_f32_32x32x16): a lane then holds, for
//           ITS query, 16 keys of every 32-key block, so the Softmax over the keys
//           is a reduction inside the lane plus one exchange with lane + 32;
//           scores, mask and exponentials stay fp32 in registers;
//   context C[dv][query] = v^T . p^T: the probabilities a lane holds are packed to
//           the operand type as they are - the order of the keys inside one MFMA
//           is free as long as v^T is stored in the same order, which the
//           transposing LDS write takes care of (slot_of_key);
//   result  rows of 64 values leave as 16-byte vectors formed by exchanging
//           dwords between lanes l and l + 32 (v_permlane32_swap).
#include "igemm_common.h"

#include <cstdlib>

namespace ohip {

namespace {

constexpr int kAttnD = 64;            // head size
constexpr float kLog2e = 1.44269504f;  // scores and mask are kept in units of log 2: the hardware exponential takes them as they are
constexpr int kKPitch = 144;          // bytes per staged k row (128 + 16: conflict-free 16-byte fragment reads)
constexpr int kVPitch = 272;          // bytes per staged v^T row (128 keys x 2 + 16)

__device__ __forceinline__ void swap32f(float& x, float& y) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uintx2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r.x);
  y = __uint_as_float(r.y);
#endif
}
__device__ __forceinline__ void swap32u(unsigned& x, unsigned& y) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uintx2 r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r.x;
  y = r.y;
#endif
}
// the value of the partner lane (l ^ 32) combined with the own one
__device__ __forceinline__ float pair_max(float v) {
  float x = v, y = v;
  swap32f(x, y);   // x = [v.lo | v.lo], y = [v.hi | v.hi]
  return fmaxf(x, y);
}
__device__ __forceinline__ float pair_sum(float v) {
  float x = v, y = v;
  swap32f(x, y);
  return x + y;
}

// Position of key (0 .. 127) inside a staged v^T row.  In the score layout a lane of half
// s holds keys kb*32 + q*8 + s*4 + r; the context product consumes, per step (kb, h), the
// lane's groups q = 2h and 2h + 1, so those eight keys sit next to each other:
// slot = kb*32 + h*16 + s*8 + (q & 1)*4 + r.
__device__ __forceinline__ int slot_of_key(const int key) {
  const int kb = key >> 5, q = (key >> 3) & 3, s = (key >> 2) & 1, r = key & 3;
  return kb * 32 + (q >> 1) * 16 + s * 8 + (q & 1) * 4 + r;
}

// The 64-byte groups of v^T row `row` (0 .. 63) lie at their places XOR this.
__device__ __forceinline__ int vt_group(const int row) { return ((row >> 3) & 3) << 6; }

// NKB: 32-key blocks of a tile; QW: wavefronts of a group, 32 queries each; LOOP: more than one tile; KG: groups that
// share the tiles.
template <typename T, int NKB, int QW, bool LOOP, int KG>
__global__ void __launch_bounds__(QW * KG * 64, 2)
attention_kernel(const AttentionParams p) {
  constexpr int TS = NKB * 32, QS = QW * 32, NT = QW * 64;
  constexpr int TILE = TS * kKPitch + kAttnD * kVPitch + TS * 4;
  static_assert(KG == 1 || KG * TILE >= QW * 34 * 256, "room for the second group's maxima, sums and contexts");
  __shared__ __attribute__((aligned(16))) unsigned char smem[KG * TILE];
  const int group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  unsigned char* ks = smem + group * TILE;
  unsigned char* vts = ks + TS * kKPitch;
  float* ms = reinterpret_cast<float*>(vts + kAttnD * kVPitch);

  const int tid = threadIdx.x - group * NT, wave = tid >> 6, lane = tid & 63;
  const int l32 = lane & 31, lg = lane >> 5;
  const int S = p.S;
  const int q_tiles = LOOP ? (S + QS - 1) / QS : 1;
  const int bh = blockIdx.x / q_tiles, qt = blockIdx.x - bh * q_tiles;
  const int b = bh / p.heads, h = bh - b * p.heads;
  const int query = qt * QS + wave * 32 + l32;   // (may lie behind the last one: computed from the last row, never stored)
  const T* q = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.q_bs + (int64_t)h * p.q_hs;
  const T* k = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.k_bs + (int64_t)h * p.k_hs;
  const T* v = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.v_bs + (int64_t)h * p.v_hs;

  // ---- this lane's piece of the query operand: d values [16 kk + 8 lg, +8) of its query
  uintx4 qf[4];
  {
    const uintx4* row = reinterpret_cast<const uintx4*>(q + (int64_t)(query < S ? query : S - 1) * p.q_rs) + lg;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[kk] = row[2 * kk];
  }
  // ---- a tile of k and v rows and mask values: requested into registers, parked in LDS.  Keys
  // behind the last one are zero rows with the mask value -inf.
  // A thread takes one 16-byte chunk of four neighbouring keys, which are neighbours in a v^T row too: eight
  // stores of 8 bytes, in a wavefront 64 bytes of each of 8 rows of each chunk, and the 64-byte groups of a row
  // change places with its number so that these fall into all banks (as 2-byte stores, 32 a thread and eight lanes
  // to a bank, the transposition was most of the launch).
  const int c = tid & 7, key4 = (tid >> 3) * 4;
  const bool stages = NT == TS * 2 || key4 < TS;   // (three blocks of keys, four wavefronts)
  constexpr int RPT = TS * 8 / NT;   // k rows of a thread, NT / 8 apart
  uintx4 kr[RPT], vr[4];
  float mr = 0.f;
  auto request = [&](const int key0) __attribute__((always_inline)) {
    const uintx4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int row = key0 + (tid >> 3) + i * (NT / 8);
      const uintx4 kv = *(reinterpret_cast<const uintx4*>(k + (int64_t)(row < S ? row : S - 1) * p.k_rs) + c);
      kr[i] = row < S ? kv : zero;
    }
    if (stages) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = key0 + key4 + i;
        const uintx4 vv = *(reinterpret_cast<const uintx4*>(v + (int64_t)(row < S ? row : S - 1) * p.v_rs) + c);
        vr[i] = row < S ? vv : zero;
      }
    }
    if (tid < TS) {
      const int key = key0 + tid;
      mr = key < S ? 0.f : -INFINITY;
      if (p.mask != nullptr && key < S) {
        if (p.mask_dt == DT_F32) mr = reinterpret_cast<const float*>(p.mask)[(int64_t)b * p.mask_bs + key];
        else mr = Store<T>::ld(reinterpret_cast<const T*>(p.mask) + (int64_t)b * p.mask_bs + key);
      }
    }
  };
  // k rows of 128 bytes, padded; v^T with the keys in slot order; the mask as fp32
  auto park = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RPT; ++i) *reinterpret_cast<uintx4*>(ks + ((tid >> 3) + i * (NT / 8)) * kKPitch + c * 16) = kr[i];
    if (stages) {
      unsigned char* dst = vts + c * 8 * kVPitch + ((slot_of_key(key4) * 2) ^ vt_group(c * 8));
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const unsigned k0 = vr[0][w], k1 = vr[1][w], k2 = vr[2][w], k3 = vr[3][w];
        *reinterpret_cast<uintx2*>(dst + (2 * w) * kVPitch) = uintx2{__builtin_amdgcn_perm(k1, k0, 0x05040100u), __builtin_amdgcn_perm(k3, k2, 0x05040100u)};
        *reinterpret_cast<uintx2*>(dst + (2 * w + 1) * kVPitch) = uintx2{__builtin_amdgcn_perm(k1, k0, 0x07060302u), __builtin_amdgcn_perm(k3, k2, 0x07060302u)};
      }
    }
    if (tid < TS) {
      // Mask values beyond 2^126 keep their order and stay finite: whatever such values differ by decides alone, and a
      // row of nothing but the type's lowest value is a plain mean.
      const float far = 0x1p+126f, m = __builtin_fabsf(mr);
      ms[tid] = m < far ? mr * kLog2e : __builtin_copysignf(__builtin_fmaf(m, 0.5f, far), mr);
    }
  };

  const float scale = p.scale * kLog2e;
  floatx16 o[2];
#pragma unroll
  for (int dvb = 0; dvb < 2; ++dvb)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dvb][e] = 0.f;
  float run_max = -INFINITY, run_sum = 0.f;

  // (both groups walk as often as the first, whose share is the longer one: a tile behind the last key holds
  // nothing but keys with the mask value -inf)
  request(group * TS);
  for (int t0 = 0; LOOP ? t0 < S : t0 == 0; t0 += KG * TS) {
    if (LOOP && t0 > 0) __syncthreads();   // everyone has used the tile before
    park();
    __syncthreads();
    if (LOOP && t0 + KG * TS < S) request(t0 + KG * TS + group * TS);

    // ---- scores: acc[kb][q*4 + r] = k[kb*32 + q*8 + lg*4 + r] . q[query]
    floatx16 acc[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[kb][e] = 0.f;
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const uintx4 a = *reinterpret_cast<const uintx4*>(ks + (kb * 32 + l32) * kKPitch + kk * 32 + lg * 16);
        acc[kb] = Mma<T>::run(a, qf[kk], acc[kb]);
      }
    // ---- Softmax over the keys of this lane's query (fp32)
    float mx = run_max;
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        const floatx4 m4 = *reinterpret_cast<const floatx4*>(ms + kb * 32 + qq * 8 + lg * 4);
        acc[kb][qq * 4 + 0] = __builtin_fmaf(acc[kb][qq * 4 + 0], scale, m4.x);
        acc[kb][qq * 4 + 1] = __builtin_fmaf(acc[kb][qq * 4 + 1], scale, m4.y);
        acc[kb][qq * 4 + 2] = __builtin_fmaf(acc[kb][qq * 4 + 2], scale, m4.z);
        acc[kb][qq * 4 + 3] = __builtin_fmaf(acc[kb][qq * 4 + 3], scale, m4.w);
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, acc[kb][qq * 4 + r]);
      }
    mx = pair_max(mx);
    // (a tile whose keys are all masked with -inf must not turn the running values into NaN)
    const float ref = LOOP && mx == -INFINITY ? 0.f : mx;
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        // (the result keeps 8 or 11 significant bits: the hardware exponential, 1 ulp, stands in for the library's)
        const float ex = __builtin_amdgcn_exp2f(acc[kb][e] - ref);
        acc[kb][e] = ex;
        sum += ex;
      }
    sum = pair_sum(sum);
    float inv = 1.f;
    if constexpr (LOOP) {
      // what the tiles before contributed, in terms of the new maximum
      const float keep = __builtin_amdgcn_exp2f(run_max - ref);
      run_sum = __builtin_fmaf(run_sum, keep, sum);
      run_max = mx;
#pragma unroll
      for (int dvb = 0; dvb < 2; ++dvb)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dvb][e] *= keep;
    } else {
      inv = 1.0f / sum;
    }

    // ---- context: o[dvb][q*4 + r] = sum over keys p[key] * v[key][dvb*32 + q*8 + lg*4 + r]
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        float pv[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pv[r] = LOOP ? acc[kb][(2 * hh) * 4 + r] : acc[kb][(2 * hh) * 4 + r] * inv;
          pv[4 + r] = LOOP ? acc[kb][(2 * hh + 1) * 4 + r] : acc[kb][(2 * hh + 1) * 4 + r] * inv;
        }
        const uintx4 pf = pack8_rne<T>(pv);
#pragma unroll
        for (int dvb = 0; dvb < 2; ++dvb) {
          const int row = dvb * 32 + l32;
          const uintx4 a = *reinterpret_cast<const uintx4*>(vts + row * kVPitch + (((kb * 32 + hh * 16 + lg * 8) * 2) ^ vt_group(row)));
          o[dvb] = Mma<T>::run(a, pf, o[dvb]);
        }
      }
  }
  if constexpr (LOOP && KG == 1) {
    const float inv = 1.0f / run_sum;
#pragma unroll
    for (int dvb = 0; dvb < 2; ++dvb)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dvb][e] *= inv;
  }
  if constexpr (KG > 1) {
    // the second group's part, a lane's values 64 places apart
    float* part = reinterpret_cast<float*>(smem) + wave * (34 * 64) + lane;
    __syncthreads();
    if (group == 1) {
#pragma unroll
      for (int dvb = 0; dvb < 2; ++dvb)
#pragma unroll
        for (int e = 0; e < 16; ++e) part[(dvb * 16 + e) * 64] = o[dvb][e];
      part[32 * 64] = run_max;
      part[33 * 64] = run_sum;
    }
    __syncthreads();
    if (group == 1) return;
    const float other_max = part[32 * 64], mx = fmaxf(run_max, other_max);
    const float ref = mx == -INFINITY ? 0.f : mx;
    float mine = __builtin_amdgcn_exp2f(run_max - ref), other = __builtin_amdgcn_exp2f(other_max - ref);
    const float inv = 1.0f / __builtin_fmaf(run_sum, mine, part[33 * 64] * other);
    mine *= inv;
    other *= inv;
#pragma unroll
    for (int dvb = 0; dvb < 2; ++dvb)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dvb][e] = __builtin_fmaf(part[(dvb * 16 + e) * 64], other, o[dvb][e] * mine);
  }

  // ---- result rows: lane (query, lg) holds, per 32-value block, the groups (q, lg) of four
  // values; after the exchange lg = 0 holds values 0 .. 15 of the block and lg = 1 16 .. 31.
  T* orow = reinterpret_cast<T*>(p.out) + (int64_t)b * p.o_bs + (int64_t)h * p.o_hs + (int64_t)(query < S ? query : S - 1) * p.o_rs;
#pragma unroll
  for (int dvb = 0; dvb < 2; ++dvb) {
    unsigned g[4][2];   // group q as two dwords (four 16-bit values)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      float f[8] = {o[dvb][qq * 4 + 0], o[dvb][qq * 4 + 1], o[dvb][qq * 4 + 2], o[dvb][qq * 4 + 3], 0.f, 0.f, 0.f, 0.f};
      const uintx4 pk = pack8_rne<T>(f);
      g[qq][0] = pk.x;
      g[qq][1] = pk.y;
    }
    // swap32(x = group q0, y = group q2): x' = [(q0, 0) | (q2, 0)], y' = [(q0, 1) | (q2, 1)]
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      swap32u(g[0][w], g[2][w]);
      swap32u(g[1][w], g[3][w]);
    }
    // now, for lg = 0: g[0] = (q0,0), g[2] = (q0,1), g[1] = (q1,0), g[3] = (q1,1): values 0 .. 15;
    // for lg = 1 the same registers hold q2 and q3: values 16 .. 31
    uintx4* dst = reinterpret_cast<uintx4*>(orow + dvb * 32 + lg * 16);
    if (query < S) {
      dst[0] = uintx4{g[0][0], g[0][1], g[2][0], g[2][1]};
      dst[1] = uintx4{g[1][0], g[1][1], g[3][0], g[3][1]};
    }
  }
}

}  // namespace

bool attention_supported(const AttentionParams& p) {
  if (const char* off = getenv("ODLA_HIP_FUSED_ATTENTION")) {   // tuning / test aid: "0" turns the kernel off
    if (off[0] == '0') return false;
  }
  if (p.dt != DT_BF16 && p.dt != DT_F16) return false;
  if (p.d != kAttnD || p.S < 1) return false;
  const int64_t q_tiles = p.S > 128 ? (p.S + 127) / 128 : 1;
  if (p.B <= 0 || p.heads <= 0 || (int64_t)p.B * p.heads * q_tiles > 0x7fffffff) return false;
  if (p.mask_dt != p.dt && p.mask_dt != DT_F32) return false;
  // rows and bases allow 16-byte accesses
  auto ok8 = [](int64_t s) { return s % 8 == 0; };
  if (!ok8(p.q_bs) || !ok8(p.q_hs) || !ok8(p.q_rs) || !ok8(p.k_bs) || !ok8(p.k_hs) || !ok8(p.k_rs) || !ok8(p.v_bs) ||
      !ok8(p.v_hs) || !ok8(p.v_rs) || !ok8(p.o_bs) || !ok8(p.o_hs) || !ok8(p.o_rs))
    return false;
  return true;
}

hipError_t launch_attention(const AttentionParams& p, hipStream_t stream) {
  if (!attention_supported(p) || p.q == nullptr || p.k == nullptr || p.v == nullptr || p.out == nullptr)
    return hipErrorInvalidValue;
  auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
  if (!al16(p.q) || !al16(p.k) || !al16(p.v) || !al16(p.out)) return hipErrorInvalidValue;
  // More than 128 keys: 128 queries a workgroup.  Where every workgroup has two compute units' worth of room, two groups, in tiles of
  // 96 keys where the longer share is then shorter than in tiles of 128.
  const int64_t q_tiles = p.S > 128 ? (p.S + 127) / 128 : 1, workgroups = (int64_t)p.B * p.heads * q_tiles;
  const auto share = [&](const int ts) { return (p.S + 2 * ts - 1) / (2 * ts) * ts; };
  const int nkb = p.S <= 128 ? (p.S + 31) / 32 : workgroups > 128 ? 5 : share(96) < share(128) ? 7 : 6;
  const dim3 grid((unsigned)workgroups);
#define ATTN_CASE(T_, CASE_, NKB_, QW_, LOOP_, KG_)                                                        \
  if (nkb == CASE_) {                                                                                      \
    hipLaunchKernelGGL((attention_kernel<T_, NKB_, QW_, LOOP_, KG_>), grid, dim3(QW_ * KG_ * 64), 0, stream, p); \
    return hipGetLastError();                                                                              \
  }
#define ATTN_CASES(T_)                                                                                     \
  ATTN_CASE(T_, 1, 1, 1, false, 1) ATTN_CASE(T_, 2, 2, 2, false, 1) ATTN_CASE(T_, 3, 3, 3, false, 1) ATTN_CASE(T_, 4, 4, 4, false, 1) \
  ATTN_CASE(T_, 5, 4, 4, true, 1) ATTN_CASE(T_, 6, 4, 4, true, 2) ATTN_CASE(T_, 7, 3, 4, true, 2)
  if (p.dt == DT_BF16) {
    ATTN_CASES(bf16_t)
  } else {
    ATTN_CASES(f16_t)
  }
#undef ATTN_CASES
#undef ATTN_CASE
  return hipErrorInvalidValue;
}

}  // namespace ohip
