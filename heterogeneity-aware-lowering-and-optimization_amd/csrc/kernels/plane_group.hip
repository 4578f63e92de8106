// Operators that stay within one plane (image, channel) of a row-major tensor, as one launch: what
// stands between convolutions, or alone, in a vision graph - BatchNorm, activations, same-shape
// arithmetic, pooling, nearest resizing, global means, channel Concats as places to store to.
//
// Launched one by one these operators are HBM-bound passes over the same few tensors, and
// channels-last pooling puts a layout change at either end.  A plane fits the LDS of a compute unit:
// a workgroup takes one plane (or several neighbouring ones, where they are small), reads the
// arguments (again, from the caches, where an element-wise instruction does), keeps in LDS what a
// later window reads, and writes each result once in the type it leaves the plan in.  BatchNorm -
// LeakyReLU - {MaxPool 3x3/2 - Resize; + x; AveragePool 2x2 - mean} - Concat on [64, 96, 75, 75] fp16,
// whose floor is 80 us (415 MB): ten launches of 341 us -> one of 116 us (3.5 TB/s; vector instructions
// take 70 us of it).  Results of the plan leave with non-temporal stores, 8 - 14 % of the whole at
// every size from 4 to 276 MB: otherwise they push the arguments that are read again out of the L2.
//
// The instructions are interpreted, which costs a scalar branch per instruction and workgroup: the
// loops over the plane are compiled per kind (and per window for the usual pools).  Four elements
// per thread and step: neighbours in the chunk for element-wise instructions (16-byte requests at
// whatever alignment the plane has), neighbours in a row for windows, which share the columns they
// read.  Element-wise instructions of equal shape give an element to the same thread, so no barrier
// stands between them.
#include "device_utils.h"

namespace ohip {

namespace {

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));       // 16 bytes at any element
typedef uint16_t ushort4u __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ float plane_bin(float a, float b, int op) {
  switch (op) {
    case BIN_ADD: return a + b;
    case BIN_SUB: return a - b;
    case BIN_MUL: return a * b;
    case BIN_DIV: return a / b;
    case BIN_MAX: return fmaxf(a, b);
    default: return fminf(a, b);
  }
}

// n / d for n < 2^20 with inv = 1 / d rounded to float: (n + 1/2) / d is 1 / (2 d) away from the next
// integer, and both roundings together move it by less than n / d / 2^23 (three full-rate instructions;
// the multiplications of fast_div run at a quarter of that).
__device__ __forceinline__ int quot(const int n, const float inv) { return (int)(((float)n + 0.5f) * inv); }

template <typename T> __device__ __forceinline__ float rounded(float v) {
  if constexpr (sizeof(T) == 4) return v;
  T t;
  Store<T>::st(&t, v);
  return Store<T>::ld(&t);
}

// Up to four elements from outside: requested (raw), then as values of type T.  base is the same for
// the whole workgroup, `at` small.
template <typename T>
__device__ __forceinline__ void ext_request4(const char* base, const DType dt, const unsigned at, const int cnt, uintx4& q) {
  if (dt == DT_F32) {
    const float* s = reinterpret_cast<const float*>(base);
    if (cnt == 4) q = __builtin_bit_cast(uintx4, *reinterpret_cast<const float4u*>(s + at));
    else {
#pragma unroll
      for (unsigned e = 0; e < 3; ++e)
        if ((int)e < cnt) q[e] = __float_as_uint(s[at + e]);
    }
  } else if constexpr (sizeof(T) == 2) {   // (the plan's own type)
    const uint16_t* s = reinterpret_cast<const uint16_t*>(base);
    if (cnt == 4) {
      const uintx2 t = __builtin_bit_cast(uintx2, *reinterpret_cast<const ushort4u*>(s + at));
      q.x = t.x;
      q.y = t.y;
    } else {
      if (cnt > 0) q.x = s[at];
      if (cnt > 1) q.x |= (unsigned)s[at + 1] << 16;
      if (cnt > 2) q.y = s[at + 2];
    }
  }
}
template <typename T>
__device__ __forceinline__ void ext_values4(const DType dt, const uintx4 q, float (&v)[4]) {
  if (dt == DT_F32) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = rounded<T>(__uint_as_float(q[e]));
  } else if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const T t = {(uint16_t)(q[e >> 1] >> (16 * (e & 1)))};
      v[e] = Store<T>::ld(&t);
    }
  }
}
template <typename T>
__device__ __forceinline__ void ext_store4(char* base, const DType dt, const int stream, const unsigned at, const int cnt, const float (&v)[4]) {
  if (dt == DT_F32) {
    float* d = reinterpret_cast<float*>(base);
    const float4u q = {v[0], v[1], v[2], v[3]};
    if (cnt == 4 && stream) __builtin_nontemporal_store(q, reinterpret_cast<float4u*>(d + at));
    else if (cnt == 4) *reinterpret_cast<float4u*>(d + at) = q;
    else {
#pragma unroll
      for (unsigned e = 0; e < 3; ++e)
        if ((int)e < cnt) d[at + e] = v[e];
    }
  } else if constexpr (sizeof(T) == 2) {
    uint16_t* d = reinterpret_cast<uint16_t*>(base);
    uint16_t q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      T t;
      Store<T>::st(&t, v[e]);
      q[e] = t.bits;
    }
    if (cnt == 4) *reinterpret_cast<ushort4u*>(d + at) = ushort4u{q[0], q[1], q[2], q[3]};
    else {
#pragma unroll
      for (unsigned e = 0; e < 3; ++e)
        if ((int)e < cnt) d[at + e] = q[e];
    }
  }
}

// four neighbours of an LDS buffer at a multiple of four
template <typename T> __device__ __forceinline__ void lds_load4(const T* s, float (&v)[4]) {
  struct alignas(sizeof(T) * 4) Q { T t[4]; };
  const Q q = *reinterpret_cast<const Q*>(s);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Store<T>::ld(&q.t[e]);
}
template <typename T> __device__ __forceinline__ void lds_store4(T* d, const float (&v)[4]) {
  struct alignas(sizeof(T) * 4) Q { T t[4]; };
  Q q;
#pragma unroll
  for (int e = 0; e < 4; ++e) Store<T>::st(&q.t[e], v[e]);
  *reinterpret_cast<Q*>(d) = q;
}

__device__ __forceinline__ void act4(float (&v)[4], const ActKind act, const float a, const float b) {
  switch (act) {
    case ACT_NONE: return;
    case ACT_RELU:
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
      return;
    case ACT_LEAKY:
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] : a * v[e];
      return;
    case ACT_CLAMP:
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fminf(fmaxf(v[e], a), b);
      return;
    case ACT_SIGMOID:
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = 1.0f / (1.0f + expf(-v[e]));
      return;
    default:   // ACT_TANH (plane_act_ok)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = tanhf(v[e]);
      return;
  }
}

// The launch's arguments where the hardware has them (constant memory): indexed by what an
// instruction names, an argument taken by value would be copied to scratch memory first.
using KLaunch = const __attribute__((address_space(4))) PlaneLaunch;
using KInst = const __attribute__((address_space(4))) PlaneInst;

// The chunk of planes a workgroup works on.
struct Chunk { int n, c0, np, tid, nt; };

// Where the chunk's planes of an outside tensor start (null for none)
__device__ __forceinline__ char* ext_base(KLaunch& p, const int x, const Chunk& k, const int hw) {
  if (x < 0) return nullptr;
  return reinterpret_cast<char*>(p.ext[x]) + ((int64_t)k.n * p.g.ext[x].img + p.g.ext[x].off + (int64_t)k.c0 * hw) * (p.g.ext[x].dt == DT_F32 ? 4 : 2);
}

template <typename T>
__device__ __forceinline__ void run_point(KLaunch& p, KInst& I, const Chunk& k, T* lds) {
  constexpr int U = 3;   // steps whose requests are in flight together
  const int hw = I.Ho * I.Wo, total = k.np * hw;
  const char* ea = ext_base(p, I.a_ext, k, hw);
  const char* eb = ext_base(p, I.b_ext, k, hw);
  char* ed = ext_base(p, I.dst_ext, k, hw);
  const DType da = I.a_ext >= 0 ? p.g.ext[I.a_ext].dt : DT_F32, db = I.b_ext >= 0 ? p.g.ext[I.b_ext].dt : DT_F32;
  const float* scale = I.affine >= 0 ? p.scale[I.affine] + k.c0 : nullptr;
  const float* shift = I.affine >= 0 ? p.shift[I.affine] + k.c0 : nullptr;
  for (int j0 = k.tid * 4; j0 < total; j0 += k.nt * 4 * U) {
    uintx4 qa[U], qb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * k.nt * 4, cnt = total - j < 4 ? total - j : 4;
      qa[u] = qb[u] = uintx4{0u, 0u, 0u, 0u};
      if (I.a_ext >= 0) ext_request4<T>(ea, da, (unsigned)j, cnt, qa[u]);
      if (I.b_ext >= 0) ext_request4<T>(eb, db, (unsigned)j, cnt, qb[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * k.nt * 4, cnt = total - j < 4 ? total - j : 4;
      if (cnt <= 0) break;
      float v[4], r[4];
      if (I.a_ext >= 0) ext_values4<T>(da, qa[u], v);
      else lds_load4(lds + I.a + j, v);
      if (I.affine >= 0) {
        if (k.np == 1) {   // (the same for the whole workgroup: scalar loads)
          const float s0 = scale[0], t0 = shift[0];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] * s0 + t0;
        } else {           // (a plane has four elements or more: a step touches two planes at most)
          const int pl = quot(j, I.hw_inv), rem = j - pl * hw;
          const int p1 = pl + 1 < k.np ? pl + 1 : pl;
          const float s0 = scale[pl], t0 = shift[pl], s1 = scale[p1], t1 = shift[p1];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = rem + e < hw ? v[e] * s0 + t0 : v[e] * s1 + t1;
        }
      }
      if (I.bin >= 0) {
        if (I.b_ext >= 0) ext_values4<T>(db, qb[u], r);
        else lds_load4(lds + I.b + j, r);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = plane_bin(v[e], r[e], I.bin);
      }
      act4(v, I.act, I.act_a, I.act_b);
      if (I.dst >= 0) lds_store4(lds + I.dst + j, v);
      if (I.dst_ext >= 0) ext_store4<T>(ed, p.g.ext[I.dst_ext].dt, p.g.ext[I.dst_ext].stream, (unsigned)j, cnt, v);
    }
  }
}

// Results of a window instruction: four neighbours of a row.  The last four of a row that is no
// multiple of four start further left and repeat what their neighbour computes (the same values to
// the same places), so that no request, store or column is conditional; rows of fewer than four
// (FEW) take `cnt` of them.
template <typename T, bool FEW>
__device__ __forceinline__ void row_store(KLaunch& p, KInst& I, T* lds, char* ed, const int at, const int cnt, const float (&v)[4]) {
  if (I.dst >= 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (!FEW || e < cnt) Store<T>::st(lds + I.dst + at + e, v[e]);
  }
  if (I.dst_ext >= 0) ext_store4<T>(ed, p.g.ext[I.dst_ext].dt, p.g.ext[I.dst_ext].stream, (unsigned)at, FEW ? cnt : 4, v);
}

// KW, SW > 0: window and step at compile time (KH = KW, SH = SW); the four results of a thread
// share the columns they read.  Taps outside the plane are read at the nearest position inside: for
// a maximum that position belongs to the same window (every window overlaps the plane here, see
// plane_prepare); FULL sums have none.
template <typename T, int KW, int SW, bool MAX, bool FULL>
__device__ __forceinline__ void pool_row4(KInst& I, const T* plane, const int r, const int c, float (&acc)[4]) {
  const int h0 = __mul24(r, I.sh) - I.ph, w0 = __mul24(c, I.sw) - I.pw;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = MAX ? -INFINITY : 0.f;
  int hv = 0;
  if constexpr (KW > 0 && FULL) {
    constexpr int NC = 3 * SW + KW;
    const T* at = plane + __mul24(h0, I.W) + w0;
#pragma unroll
    for (int a = 0; a < KW; ++a) {
      float v[NC];
#pragma unroll
      for (int x = 0; x < NC; ++x) v[x] = Store<T>::ld(at + x);
      at += I.W;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int s = 0; s < KW; ++s) acc[e] = acc[e] + v[e * SW + s];
    }
  } else if constexpr (KW > 0) {
    constexpr int NC = 3 * SW + KW;
    const T* row[KW];
    bool in[KW];
#pragma unroll
    for (int a = 0; a < KW; ++a) {
      const int hi = h0 + a;
      in[a] = (unsigned)hi < (unsigned)I.H;
      row[a] = plane + __mul24(hi < 0 ? 0 : (hi < I.H ? hi : I.H - 1), I.W);
      hv += in[a] ? 1 : 0;
    }
    if constexpr (MAX) {
      float m[NC];   // over a column of the window
#pragma unroll
      for (int x = 0; x < NC; ++x) {
        const int wi = w0 + x, col = wi < 0 ? 0 : (wi < I.W ? wi : I.W - 1);
        m[x] = Store<T>::ld(row[0] + col);
#pragma unroll
        for (int a = 1; a < KW; ++a) m[x] = fmaxf(m[x], Store<T>::ld(row[a] + col));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int s = 0; s < KW; ++s) acc[e] = fmaxf(acc[e], m[e * SW + s]);
    } else {
      int col[NC];
      bool ok[NC];
#pragma unroll
      for (int x = 0; x < NC; ++x) {
        const int wi = w0 + x;
        ok[x] = (unsigned)wi < (unsigned)I.W;
        col[x] = ok[x] ? wi : 0;
      }
#pragma unroll
      for (int a = 0; a < KW; ++a) {
        float v[NC];
#pragma unroll
        for (int x = 0; x < NC; ++x) {
          const float got = Store<T>::ld(row[a] + col[x]);
          v[x] = in[a] && ok[x] ? got : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int s = 0; s < KW; ++s) acc[e] = acc[e] + v[e * SW + s];
      }
    }
  } else {
    for (int a = 0; a < I.kh; ++a) {
      const int hi = h0 + a;
      if ((unsigned)hi >= (unsigned)I.H) continue;
      ++hv;
      for (int s = 0; s < I.kw; ++s) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int wi = w0 + e * I.sw + s;
          if ((unsigned)wi < (unsigned)I.W) {
            const float got = Store<T>::ld(plane + hi * I.W + wi);
            acc[e] = MAX ? fmaxf(acc[e], got) : acc[e] + got;
          }
        }
      }
    }
  }
  if constexpr (!MAX) {
    if (I.inv != 0.f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] *= I.inv;
    } else if (I.div != 0) {
      const float d = (float)I.div;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] /= d;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int lo = w0 + e * I.sw, a = lo < 0 ? 0 : lo, b = lo + I.kw < I.W ? lo + I.kw : I.W;
        const int n = hv * (b > a ? b - a : 0);
        acc[e] /= (float)(n > 0 ? n : 1);
      }
    }
  }
}

template <typename T, int KW, int SW, bool MAX, bool FULL>
__device__ __forceinline__ void run_pool(KLaunch& p, KInst& I, const Chunk& k, T* lds, float* red) {
  const int Q = (I.Wo + 3) >> 2, per = I.Ho * Q, hw_in = I.H * I.W, hw = I.Ho * I.Wo;
  char* ed = ext_base(p, I.dst_ext, k, hw);
  constexpr bool FEW = KW == 0;   // (the usual windows: rows of four results or more, see plane_prepare)
  // four results; the first `skip` of them are a neighbour's, `cnt` exist
  auto unit = [&](const int pl, const int i, float (&v)[4], int& skip, int& cnt) __attribute__((always_inline)) {
    const int r = quot(i, I.q_inv), c4 = (i - __mul24(r, Q)) * 4;
    const int c = FEW || c4 + 4 <= I.Wo ? c4 : I.Wo - 4;
    skip = c4 - c;
    cnt = FEW && I.Wo - c < 4 ? I.Wo - c : 4;
    pool_row4<T, KW, SW, MAX, FULL>(I, lds + I.a + __mul24(pl, hw_in), r, c, v);
    row_store<T, FEW>(p, I, lds, ed, __mul24(pl, hw) + __mul24(r, I.Wo) + c, cnt, v);
  };
  if (I.mean_ext < 0) {
    const int total = k.np * per;
    for (int i = k.tid; i < total; i += k.nt) {
      const int pl = k.np == 1 ? 0 : quot(i, I.rq_inv);
      float v[4];
      int skip, cnt;
      unit(pl, i - __mul24(pl, per), v, skip, cnt);
    }
    return;
  }
  if constexpr (!MAX) {
    // plane means: a wavefront per plane, or the whole workgroup where there are fewer planes
    const auto& x = p.g.ext[I.mean_ext];
    const int64_t em = (int64_t)k.n * x.img + x.off + k.c0;
    const int lane = k.tid & 63, wave = k.tid >> 6, waves = k.nt >> 6;
    const bool by_wave = k.np >= waves;
    for (int pl = by_wave ? wave : 0; pl < k.np; pl += by_wave ? waves : 1) {
      float s = 0.f;
      for (int i = by_wave ? lane : k.tid; i < per; i += by_wave ? 64 : k.nt) {
        float v[4];
        int skip, cnt;
        unit(pl, i, v, skip, cnt);
#pragma unroll
        for (int e = 0; e < 4; ++e) s += e >= skip && e < cnt ? rounded<T>(v[e]) : 0.f;
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d);
      if (!by_wave) {
        if (lane == 0) red[wave] = s;
        __syncthreads();
        s = 0.f;
        for (int w = 0; w < waves; ++w) s += red[w];
        __syncthreads();   // (red is written again for the next plane)
      }
      if (by_wave ? lane == 0 : k.tid == 0) {
        const float m = s / (float)hw;
        if (x.dt == DT_F32) reinterpret_cast<float*>(p.ext[I.mean_ext])[em + pl] = m;
        else if constexpr (sizeof(T) == 2) Store<T>::st(reinterpret_cast<T*>(p.ext[I.mean_ext]) + em + pl, m);
      }
    }
  }
}

template <typename T>
__device__ __forceinline__ void run_resize(KLaunch& p, KInst& I, const Chunk& k, T* lds) {
  const int Q = (I.Wo + 3) >> 2, per = I.Ho * Q, hw_in = I.H * I.W, hw = I.Ho * I.Wo, total = k.np * per;
  char* ed = ext_base(p, I.dst_ext, k, hw);
  for (int i = k.tid; i < total; i += k.nt) {
    const int pl = k.np == 1 ? 0 : quot(i, I.rq_inv), rem = i - __mul24(pl, per);
    const int r = quot(rem, I.q_inv), c4 = (rem - __mul24(r, Q)) * 4;
    const int c = c4 + 4 <= I.Wo ? c4 : (I.Wo > 4 ? I.Wo - 4 : 0), cnt = I.Wo - c < 4 ? I.Wo - c : 4;
    const T* row = lds + I.a + __mul24(pl, hw_in) + __mul24(quot(__mul24(r, I.H), I.ho_inv), I.W);
    const float t0 = (float)__mul24(c, I.W) + 0.5f, step = (float)I.W;   // (whole numbers and a half: exact)
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int wi = (int)((t0 + (float)e * step) * I.wo_inv);   // quot((c + e) * W)
      v[e] = Store<T>::ld(row + (wi < I.W ? wi : I.W - 1));      // (behind the end of a row of fewer than four)
    }
    row_store<T, true>(p, I, lds, ed, __mul24(pl, hw) + __mul24(r, I.Wo) + c, cnt, v);
  }
}

template <typename T>
__global__ void __launch_bounds__(1024) plane_group_kernel(const PlaneLaunch) {
#if defined(__HIP_DEVICE_COMPILE__)
  KLaunch& p = *(KLaunch*)__builtin_amdgcn_kernarg_segment_ptr();
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float red[16];
  T* lds = reinterpret_cast<T*>(smem);
  Chunk k;
  k.n = fast_div(blockIdx.x, p.g.chunk_magic, p.g.chunk_shift);
  k.c0 = ((int)blockIdx.x - k.n * p.g.chunks) * p.g.planes;
  k.np = p.g.C - k.c0 < p.g.planes ? p.g.C - k.c0 : p.g.planes;
  k.tid = threadIdx.x;
  k.nt = p.g.threads;
  for (int ii = 0; ii < p.g.n_inst; ++ii) {   // (uniform: every thread runs every instruction)
    KInst& I = p.g.inst[ii];
    if (I.barrier) __syncthreads();
    if (I.kind == PLANE_POINT) {
      run_point<T>(p, I, k, lds);
    } else if (I.kind == PLANE_RESIZE) {
      run_resize<T>(p, I, k, lds);
    } else {
      switch (I.window) {
#define POOL_CASE(N_, KW_, SW_, MAX_, FULL_) case N_: run_pool<T, KW_, SW_, MAX_, FULL_>(p, I, k, lds, red); break
        POOL_CASE(1, 1, 1, false, true);
        POOL_CASE(2, 2, 1, false, true);
        POOL_CASE(3, 2, 2, false, true);
        POOL_CASE(4, 3, 2, false, false);
        POOL_CASE(5, 2, 2, true, false);
        POOL_CASE(6, 3, 2, true, false);
        POOL_CASE(7, 3, 1, true, false);
        POOL_CASE(8, 0, 0, true, false);
        default: run_pool<T, 0, 0, false, false>(p, I, k, lds, red); break;
#undef POOL_CASE
      }
    }
  }
#endif
}

}  // namespace

bool plane_act_ok(ActKind a) {
  return a == ACT_NONE || a == ACT_RELU || a == ACT_LEAKY || a == ACT_CLAMP || a == ACT_SIGMOID || a == ACT_TANH;
}

void plane_prepare(PlaneGroup* g) {
  div_magic(g->chunks, &g->chunk_magic, &g->chunk_shift);
  for (int i = 0; i < g->n_inst; ++i) {
    PlaneInst& I = g->inst[i];
    const int q = (I.Wo + 3) / 4;
    I.hw_inv = 1.0f / (float)(I.Ho * I.Wo);
    I.rq_inv = 1.0f / (float)(I.Ho * q);
    I.q_inv = 1.0f / (float)q;
    I.ho_inv = 1.0f / (float)I.Ho;
    I.wo_inv = 1.0f / (float)I.Wo;
    if (I.kind != PLANE_POOL) continue;
    // (size and step as one number, for those that have a compiled window: single digits only)
    const int ks = I.kh == I.kw && I.sh == I.sw && I.kh <= 3 && I.sh <= 2 ? I.kh * 10 + I.sh : 0;
    const bool full = I.ph == 0 && I.pw == 0 && (I.Ho - 1) * I.sh + I.kh <= I.H && (I.Wo - 1) * I.sw + I.kw <= I.W;
    const bool overlap = I.ph < I.kh && I.pw < I.kw && (I.Ho - 1) * I.sh - I.ph < I.H && (I.Wo - 1) * I.sw - I.pw < I.W;
    I.window = I.is_max ? (!overlap ? 8 : ks == 22 ? 5 : ks == 32 ? 6 : ks == 31 ? 7 : 8)
                        : (ks == 32 ? 4 : !full ? 9 : ks == 11 ? 1 : ks == 21 ? 2 : ks == 22 ? 3 : 9);
    if (I.Wo < 4) I.window = I.is_max ? 8 : 9;
    const int n = I.kh * I.kw;
    I.div = I.count_pad || full ? n : 0;
    I.inv = I.div != 0 && (n & (n - 1)) == 0 ? 1.0f / (float)n : 0.f;   // (a power of two: the same result)
  }
}

// What a launch takes, in microseconds: the longer of the instructions of one workgroup that has a
// compute unit to itself, of all workgroups of a unit at the rate their threads share, and of the traffic.
// A step is four elements of every thread.  Fitted to 154 calls that are one chain (1 .. 16384 planes of
// 14 x 14 .. 230 x 230, fp16 and fp32): with 12 us for the call around the launch, 95 % of them are within 20 %.
float plane_group_us(const PlaneGroup& g) {
  const float full = (float)g.threads / 1024.f, alone = 0.55f + 0.45f * full;   // (few wavefronts hide less, but share less)
  float chain = 0.f, shared = 0.f, bytes = 0.f;
  for (int i = 0; i < g.n_inst; ++i) {
    const PlaneInst& I = g.inst[i];
    const float units = (float)g.planes * (I.kind == PLANE_POINT ? (float)I.Ho * I.Wo / 4.f : (float)I.Ho * ((I.Wo + 3) / 4));
    const float steps = units / (float)g.threads;
    const bool loop = I.kind == PLANE_POOL && I.window >= 8;   // a window that is not compiled: a chain of reads, tap after tap
    const float us = loop ? 0.25f * (float)I.kh * (float)I.kw
                          : I.kind == PLANE_POOL ? 0.2f + 0.12f * (float)I.kh * (float)I.kw
                                                 : I.kind == PLANE_RESIZE ? 0.47f : 0.55f + (I.act == ACT_SIGMOID || I.act == ACT_TANH ? 0.9f : 0.f);
    chain += 0.3f + (loop ? ceilf(steps) * us : steps * us * alone);
    shared += steps * us * full * (loop ? 1.f : 0.7f);
    for (int x : {I.a_ext, I.b_ext, I.dst_ext})
      if (x >= 0) bytes += (float)g.N * (float)g.C * (float)g.ext[x].hw * (g.ext[x].dt == DT_F32 ? 4.f : 2.f);
  }
  const float per_unit = ceilf((float)g.N * (float)g.chunks / 256.f);
  return 2.f + fmaxf(fmaxf(chain, shared * per_unit), bytes / 3.5e6f);
}

hipError_t launch_plane_group(const PlaneLaunch& l, hipStream_t stream) {
  const PlaneGroup& g = l.g;
  for (int i = 0; i < g.n_inst && i < kPlaneMaxInst; ++i)   // (means are of averages: run_pool)
    if (g.inst[i].mean_ext >= 0 && (g.inst[i].kind != PLANE_POOL || g.inst[i].is_max)) return hipErrorInvalidValue;
  if (g.n_inst <= 0 || g.n_inst > kPlaneMaxInst || g.N <= 0 || g.C <= 0 || g.planes <= 0 || g.threads < 64 || g.threads > 1024 ||
      g.lds_bytes > kPlaneLdsMax || (int64_t)g.N * g.chunks > 0x7fffffff || (int64_t)g.planes * g.chunks < g.C)
    return hipErrorInvalidValue;
  static_assert(sizeof(PlaneLaunch) <= 4096, "kernel arguments");
  const dim3 grid((unsigned)(g.N * g.chunks));
#define PLANE_GO(T_)                                                                                       \
  do {                                                                                                     \
    if (g.lds_bytes > 64 * 1024) {                                                                         \
      static LdsLimit limit;                                                                               \
      const hipError_t e = limit.raise(reinterpret_cast<const void*>(plane_group_kernel<T_>), kPlaneLdsMax); \
      if (e != hipSuccess) return e;                                                                       \
    }                                                                                                      \
    hipLaunchKernelGGL(plane_group_kernel<T_>, grid, dim3(g.threads), g.lds_bytes, stream, l);             \
  } while (0)
  switch (g.dt) {
    case DT_F32: PLANE_GO(float); break;
    case DT_F16: PLANE_GO(f16_t); break;
    case DT_BF16: PLANE_GO(bf16_t); break;
    default: return hipErrorInvalidValue;
  }
#undef PLANE_GO
  return hipGetLastError();
}

}  // namespace ohip
