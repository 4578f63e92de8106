// Streaming element-wise kernels for gfx950: unary activations, per-channel
// affine (folded BatchNorm), broadcasting binary ops, casts and affine
// (de)quantisation.  All are HBM-bound: each thread moves 16-byte vectors,
// consecutive lanes touch consecutive vectors, and the grid is a grid-stride
// loop sized to a few workgroups per CU.
#include "device_utils.h"

namespace ohip {

namespace {
constexpr int kThreads = 256;

// Streaming loop shape shared by the flat kernels: every thread keeps U 16-byte
// loads in flight before it touches the data.  Results leave with plain stores:
// measured on [256,256,56,56] fp16, non-temporal stores were slower here (ReLU
// 168 -> 269 us, residual Add 238 -> 252 us), unlike in the convolution epilogue.
constexpr int kUnroll = 4;

template <typename T>
__device__ __forceinline__ void out_store(Vec16<T>& v, T* p) {
  v.store(p);
}

// A workgroup owns one contiguous tile of kThreads * U 16-byte vectors: load u of
// a thread is vector tile * kThreads * U + u * kThreads + thread, so that every
// load instruction of a wavefront covers one contiguous KiB and a workgroup's U
// loads cover one contiguous U * 4 KiB, all in flight before the first use.
// KIND >= 0 fixes the activation at compile time (the switch folds away; per
// element it would cost more than the arithmetic); KIND < 0 takes it from `act`.
template <typename T, int KIND, int U>
__global__ void __launch_bounds__(kThreads)
unary_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t n, ActKind act, float a, float b) {
  constexpr int V = Vec16<T>::N;
  const ActKind kind = KIND >= 0 ? (ActKind)KIND : act;
  const int64_t nvec = n / V;
  const int64_t base = (int64_t)blockIdx.x * (kThreads * U) + threadIdx.x;
  Vec16<T> v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i < nvec) v[u].raw = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(x + i * V));
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i < nvec) {
      if constexpr (KIND == ACT_NEG) {   // (sign bits, a word at a time: see f32_to_bf16)
        v[u].raw ^= sizeof(T) == 4 ? 0x80000000u : 0x80008000u;
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) v[u].set(e, apply_act(v[u].get(e), kind, a, b));
      }
      out_store(v[u], y + i * V);
    }
  }
  // tail (fewer than V elements), by the first workgroup
  if (blockIdx.x == 0) {
    for (int64_t i = nvec * V + threadIdx.x; i < n; i += kThreads)
      Store<T>::st(y + i, apply_act(Store<T>::ld(x + i), kind, a, b));
  }
}

// y = x * scale[c] + shift[c] on row-major N,C,inner tensors (inner > 1): the channel is constant
// across a vector when inner % V == 0.  (Channels-last tensors: channel_rows_kernel.)
template <typename T, int U>
__global__ void __launch_bounds__(kThreads)
channel_affine_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t n, int64_t inner,
                      int channels, const float* __restrict__ scale,
                      const float* __restrict__ shift) {
  constexpr int V = Vec16<T>::N;
  if (inner % V == 0) {
    // tiled like unary_kernel: a workgroup owns kThreads * U consecutive vectors
    const int64_t nvec = n / V;
    const int64_t base = (int64_t)blockIdx.x * (kThreads * U) + threadIdx.x;
    Vec16<T> v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = base + u * kThreads;
      if (i < nvec) v[u].raw = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(x + i * V));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = base + u * kThreads;
      if (i >= nvec) continue;
      const int c = (int)(((i * V) / inner) % channels);
      const float sc = scale[c], sh = shift[c];
#pragma unroll
      for (int e = 0; e < V; ++e) v[u].set(e, v[u].get(e) * sc + sh);
      out_store(v[u], y + i * V);
    }
  } else {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      const int c = (int)((i / inner) % channels);
      Store<T>::st(y + i, Store<T>::ld(x + i) * scale[c] + shift[c]);
    }
  }
}

__device__ __forceinline__ float bin_op(float a, float b, BinKind op) {
  switch (op) {
    case BIN_ADD: return a + b;
    case BIN_SUB: return a - b;
    case BIN_MUL: return a * b;
    case BIN_DIV: return a / b;
    case BIN_MAX: return fmaxf(a, b);
    case BIN_MIN: return fminf(a, b);
  }
  return a;
}

// Channels-last rows (pixels) of C channels, each tensor with its own pitch:
//   y[m][c] = act((x[m][c] * scale[c] + shift[c]) op r[m][c])
// with the affine part, the operand r and the activation optional - BatchNorm with its activation,
// an element-wise operator, an activation - so that the result can be a channel slice of a wider
// tensor (the place it has in a Concat) and nothing is copied there afterwards.
// HBM-bound; one pass over what each operand holds.  W = 8 (2-byte types) or 4: vectors of W
// channels; W = 1: single elements, where the channel count or a pitch is odd.  Tiled like
// unary_kernel.  OP / KIND >= 0 fix the operator / the activation at compile time.
template <typename T, int W, bool AFFINE, int OP, int KIND, int U>
__global__ void __launch_bounds__(kThreads) channel_rows_kernel(const ChannelRowsParams p) {
  const T* x = reinterpret_cast<const T*>(p.x);
  const T* r = reinterpret_cast<const T*>(p.r);
  T* y = reinterpret_cast<T*>(p.y);
  constexpr bool kOp = OP != -2;   // -2: no second operand
  const ActKind kind = KIND >= 0 ? (ActKind)KIND : p.act;
  const BinKind op = OP >= 0 ? (BinKind)OP : p.op;
  const int cw = p.C / W;
  const int64_t n = p.rows * cw;   // (the launcher checks n < 2^31)
  const int64_t base = (int64_t)blockIdx.x * (kThreads * U) + threadIdx.x;
  struct alignas(W == 1 ? sizeof(T) : 16) Unit { T v[W]; };
  Unit vx[U], vr[U];
  int64_t m[U];
  int c[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i < n) {
      m[u] = fast_div((int)i, p.cw_magic, p.cw_shift);
      c[u] = ((int)i - (int)m[u] * cw) * W;
      vx[u] = *reinterpret_cast<const Unit*>(x + m[u] * p.xcs + c[u]);
      if constexpr (kOp) vr[u] = *reinterpret_cast<const Unit*>(r + m[u] * p.rcs + c[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i >= n) continue;
    float f[W];
#pragma unroll
    for (int e = 0; e < W; ++e) f[e] = Store<T>::ld(&vx[u].v[e]);
    if constexpr (AFFINE) {
      float sc[W], sh[W];
#pragma unroll
      for (int e = 0; e < W; ++e) { sc[e] = p.scale[c[u] + e]; sh[e] = p.shift[c[u] + e]; }
#pragma unroll
      for (int e = 0; e < W; ++e) f[e] = f[e] * sc[e] + sh[e];
    }
#pragma unroll
    for (int e = 0; e < W; ++e) {
      if constexpr (kOp) f[e] = bin_op(f[e], Store<T>::ld(&vr[u].v[e]), op);
      Store<T>::st(&vx[u].v[e], apply_act(f[e], kind, p.act_a, p.act_b));
    }
    *reinterpret_cast<Unit*>(y + m[u] * p.ycs + c[u]) = vx[u];
  }
}

__global__ void bn_fold_kernel(const float* mean, const float* var, const float* gamma,
                               const float* beta, float sgamma, float sbeta, float eps,
                               int channels, float* scale, float* shift) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const float g = gamma ? gamma[c] : sgamma;
  const float b = beta ? beta[c] : sbeta;
  const float m = g / sqrtf(var[c] + eps);
  scale[c] = m;
  shift[c] = b - mean[c] * m;
}

// Same-shape, contiguous operands; tiled like unary_kernel.  OP / KIND >= 0 fix the
// operator / the fused activation at compile time.
template <typename T, int OP, int KIND, int U>
__global__ void __launch_bounds__(kThreads)
binary_flat_kernel(const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ y, int64_t n,
                   BinKind op_rt, ActKind act, float aa, float ab) {
  constexpr int V = Vec16<T>::N;
  const BinKind op = OP >= 0 ? (BinKind)OP : op_rt;
  const ActKind kind = KIND >= 0 ? (ActKind)KIND : act;
  const int64_t nvec = n / V;
  const int64_t base = (int64_t)blockIdx.x * (kThreads * U) + threadIdx.x;
  Vec16<T> va[U], vb[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i < nvec) {
      va[u].raw = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(a + i * V));
      vb[u].raw = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(b + i * V));
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = base + u * kThreads;
    if (i < nvec) {
#pragma unroll
      for (int e = 0; e < V; ++e) va[u].set(e, apply_act(bin_op(va[u].get(e), vb[u].get(e), op), kind, aa, ab));
      out_store(va[u], y + i * V);
    }
  }
  if (blockIdx.x == 0) {
    for (int64_t i = nvec * V + threadIdx.x; i < n; i += kThreads)
      Store<T>::st(y + i, apply_act(bin_op(Store<T>::ld(a + i), Store<T>::ld(b + i), op), kind, aa, ab));
  }
}

// One operand is a vector indexed by the innermost output dim (bias rows,
// channels-last per-channel constants): b index = i % period.
template <typename T>
__global__ void __launch_bounds__(kThreads)
binary_rowvec_kernel(const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ y,
                     int64_t n, int period, bool b_is_lhs, BinKind op, ActKind act, float aa,
                     float ab) {
  constexpr int V = Vec16<T>::N;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (period % V == 0) {
    const int64_t nvec = n / V;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nvec; i += stride) {
      Vec16<T> va, vb;
      va.load(a + i * V);
      vb.load(b + (i * V) % period);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float l = b_is_lhs ? vb.get(e) : va.get(e);
        const float r = b_is_lhs ? va.get(e) : vb.get(e);
        va.set(e, apply_act(bin_op(l, r, op), act, aa, ab));
      }
      va.store(y + i * V);
    }
  } else {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      const float av = Store<T>::ld(a + i), bv = Store<T>::ld(b + i % period);
      Store<T>::st(y + i, apply_act(b_is_lhs ? bin_op(bv, av, op) : bin_op(av, bv, op), act, aa, ab));
    }
  }
}

// General broadcast: decompose the flat output index over `rank` dims.
template <typename T>
__global__ void __launch_bounds__(kThreads)
binary_bcast_kernel(BinaryParams p, int64_t n) {
  const T* a = reinterpret_cast<const T*>(p.a);
  const T* b = reinterpret_cast<const T*>(p.b);
  T* y = reinterpret_cast<T*>(p.y);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
    int64_t rem = i, oa = 0, ob = 0;
#pragma unroll
    for (int d = 5; d >= 0; --d) {
      if (d < p.rank) {
        const int64_t q = rem / p.dims[d];
        const int64_t idx = rem - q * p.dims[d];
        rem = q;
        oa += idx * p.sa[d];
        ob += idx * p.sb[d];
      }
    }
    Store<T>::st(y + i, apply_act(bin_op(Store<T>::ld(a + oa), Store<T>::ld(b + ob), p.op), p.act,
                                  p.act_a, p.act_b));
  }
}

// Quantised add (8-bit levels stored as q-128), same shape, contiguous:
// the float sequence dequantise, op, requantise of the unfused graph.
__global__ void __launch_bounds__(kThreads)
binary_q8_kernel(BinaryParams p, int64_t n) {
  const int8_t* a = reinterpret_cast<const int8_t*>(p.a);
  const int8_t* b = reinterpret_cast<const int8_t*>(p.b);
  int8_t* y = reinterpret_cast<int8_t*>(p.y);
  const int64_t nvec = n / 16;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  auto one = [&](int8_t sa, int8_t sb) -> int8_t {
    const float fa = (float)(q_from_stored(sa) - p.a_zp) * p.a_scale;
    const float fb = (float)(q_from_stored(sb) - p.b_zp) * p.b_scale;
    const float f = bin_op(fa, fb, p.op);
    int q = (int)rintf(f * p.y_inv) + p.y_zp;
    q = q < p.y_lo ? p.y_lo : q;
    q = q > 255 ? 255 : q;
    return q_to_stored(q);
  };
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nvec; i += stride) {
    uintx4 va = *reinterpret_cast<const uintx4*>(a + i * 16);
    uintx4 vb = *reinterpret_cast<const uintx4*>(b + i * 16);
    const int8_t* ea = reinterpret_cast<const int8_t*>(&va);
    const int8_t* eb = reinterpret_cast<const int8_t*>(&vb);
    uintx4 vo;
    int8_t* eo = reinterpret_cast<int8_t*>(&vo);
#pragma unroll
    for (int e = 0; e < 16; ++e) eo[e] = one(ea[e], eb[e]);
    *reinterpret_cast<uintx4*>(y + i * 16) = vo;
  }
  for (int64_t i = nvec * 16 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride)
    y[i] = one(a[i], b[i]);
}

template <typename TS, typename TD>
__global__ void __launch_bounds__(kThreads)
cast_kernel(const TS* __restrict__ x, TD* __restrict__ y, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  // 4 elements per thread step keeps loads/stores >= 8 bytes for 16-bit types.
  const int64_t n4 = n / 4;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4; i += stride) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = Store<TS>::ld(x + i * 4 + e);
#pragma unroll
    for (int e = 0; e < 4; ++e) Store<TD>::st(y + i * 4 + e, v[e]);
  }
  for (int64_t i = n4 * 4 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride)
    Store<TD>::st(y + i, Store<TS>::ld(x + i));
}

// Up to four operators with a constant each behind one conversion, every result rounded as it would be stored: what
// bounds these is the number of launches (an attention mask of 41 values: conversion, difference and product of 1.5 us
// each and the gaps behind them; an encoder of 63 launches 377.3 -> 375.3 us, 64 x 128 values 2.8 + 7.6 + 5.6 us).
template <typename TS, typename T>
__global__ void __launch_bounds__(kThreads)
scalar_chain_kernel(const TS* __restrict__ x, T* __restrict__ y, int64_t n, const ScalarChain s) {
  auto stored = [](const float v) {
    T t;
    Store<T>::st(&t, v);
    return Store<T>::ld(&t);
  };
  float c[kScalarChain];
#pragma unroll
  for (int k = 0; k < kScalarChain; ++k) c[k] = k < s.n ? stored(s.c[k]) : 0.f;
  auto value = [&](float v) {
    v = stored(v);
#pragma unroll
    for (int k = 0; k < kScalarChain; ++k)
      if (k < s.n) v = stored(s.lhs[k] ? bin_op(c[k], v, s.op[k]) : bin_op(v, c[k], s.op[k]));
    return v;
  };
  const int64_t stride = (int64_t)gridDim.x * blockDim.x, n4 = n / 4;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n4; i += stride) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = Store<TS>::ld(x + i * 4 + e);
#pragma unroll
    for (int e = 0; e < 4; ++e) Store<T>::st(y + i * 4 + e, value(v[e]));
  }
  for (int64_t i = n4 * 4 + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) Store<T>::st(y + i, value(Store<TS>::ld(x + i)));
}

// Conversions that involve an integer type, one element per thread step.
// Rules, following the reference's cast (a oneDNN reorder): a floating-point
// value that becomes an integer is rounded to the nearest integer, ties to
// even, and saturates at the ends of the target range; an integer that becomes
// a narrower integer saturates; an integer that becomes a floating-point value
// is rounded to nearest even; anything that becomes a bool is "!= 0".
// [ref: ODLA/platforms/dnnl/odla_dnnl_cast.cc:232-258]
template <typename T> struct CastElem;
template <> struct CastElem<float> { static constexpr bool is_float = true; };
template <> struct CastElem<f16_t> { static constexpr bool is_float = true; };
template <> struct CastElem<bf16_t> { static constexpr bool is_float = true; };
template <> struct CastElem<int8_t> { static constexpr bool is_float = false; static constexpr long long lo = -128, hi = 127; };
template <> struct CastElem<uint8_t> { static constexpr bool is_float = false; static constexpr long long lo = 0, hi = 255; };
template <> struct CastElem<int32_t> { static constexpr bool is_float = false; static constexpr long long lo = -2147483648ll, hi = 2147483647ll; };
template <> struct CastElem<int64_t> { static constexpr bool is_float = false; static constexpr long long lo = INT64_MIN, hi = INT64_MAX; };

// float -> integer type TD: clamp in float to the representable ends of the
// target (2147483520 is the largest float below 2^31, 2^63 - 2^39 the largest
// below 2^63), then round to nearest even.  NaN becomes 0.
template <typename TD>
__device__ __forceinline__ TD float_to_int_sat(float v) {
  if (v != v) return (TD)0;
  float lo, hi;
  if constexpr (sizeof(TD) == 8) { lo = -9223372036854775808.f; hi = 9223371487098961920.f; }
  else if constexpr (sizeof(TD) == 4) { lo = -2147483648.f; hi = 2147483520.f; }
  else { lo = (float)CastElem<TD>::lo; hi = (float)CastElem<TD>::hi; }
  const float c = fminf(fmaxf(v, lo), hi);
  if constexpr (sizeof(TD) == 8) return (TD)__float2ll_rn(c);
  else return (TD)__float2int_rn(c);
}

template <typename TS, typename TD, bool kDstBool>
__global__ void __launch_bounds__(kThreads)
cast_int_kernel(const TS* __restrict__ x, TD* __restrict__ y, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
    if constexpr (CastElem<TS>::is_float) {
      const float v = Store<TS>::ld(x + i);
      if constexpr (kDstBool) y[i] = (TD)(v != 0.f);
      else y[i] = float_to_int_sat<TD>(v);
    } else {
      const long long v = (long long)x[i];
      if constexpr (kDstBool) {
        y[i] = (TD)(v != 0);
      } else if constexpr (CastElem<TD>::is_float) {
        Store<TD>::st(y + i, (float)v);
      } else {
        const long long lo = CastElem<TD>::lo, hi = CastElem<TD>::hi;
        y[i] = (TD)(v < lo ? lo : (v > hi ? hi : v));
      }
    }
  }
}

// q = sat(rne(x / scale) + zp)
template <typename TS>
__device__ __forceinline__ int quant_one(float x, float scale, float zf, bool sgn) {
  const float t = rintf(x / scale) + zf;  // the reference adds the zero point in float before the saturating cast
  return sgn ? (int)fminf(fmaxf(t, -128.f), 127.f) : (int)fminf(fmaxf(t, 0.f), 255.f);
}

// rne(x / scale) without the division where that is certain: x * (1 / scale) is within 1.5
// units of the last place of the quotient, so unless it lies that close to a rounding boundary
// (k + 0.5) both round to the same integer; the rare lanes near a boundary divide.
__device__ __forceinline__ float rne_quotient(float x, float scale, float inv) {
  const float m = x * inv;
  float q = rintf(m);
  if (fabsf(fabsf(m - q) - 0.5f) <= 4e-7f * fabsf(m) + 1e-30f) q = rintf(x / scale);
  return q;
}

template <typename TS>
__global__ void __launch_bounds__(kThreads)
quantize_kernel(QuantParams p) {
  const TS* x = reinterpret_cast<const TS*>(p.src);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int64_t done = 0;
  if (p.channels == 1 && (reinterpret_cast<uintptr_t>(p.src) & 15u) == 0 && (reinterpret_cast<uintptr_t>(p.dst) & 15u) == 0) {
    // per-tensor parameters: a workgroup takes contiguous tiles of 256 threads x 2 x 16 elements;
    // a thread's loads are issued back to back and each of its two results is one 16-byte store
    const float sc = p.scale[0], zf = p.zp ? (float)p.zp[0] : 0.f;
    const float inv = 1.0f / sc;
    constexpr int LV = 16 * (int)sizeof(TS) / 16;   // 16-byte loads per 16 elements
    constexpr int PER = 16 / LV;                     // elements per load
    const int64_t tile = (int64_t)kThreads * 32;
    const int64_t ntiles = p.n / tile;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
      Vec16<TS> in[2][LV];
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int l = 0; l < LV; ++l) in[g][l].load(x + t * tile + ((int64_t)g * kThreads + threadIdx.x) * 16 + l * PER);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        uintx4 ov;
        if (!p.dst_signed) {
          // unsigned levels: the packing conversion rounds (an integer already) and saturates to [0, 255]
          unsigned w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
          for (int l = 0; l < LV; ++l)
#pragma unroll
            for (int e = 0; e < PER; ++e) {
              const int k = l * PER + e;
              w[k >> 2] = __builtin_amdgcn_cvt_pk_u8_f32(rne_quotient(in[g][l].get(e), sc, inv) + zf, k & 3, w[k >> 2]);
            }
          const unsigned flip = p.dst_dt == DT_I8 ? 0x80808080u : 0u;   // stored as level - 128
          ov = uintx4{w[0] ^ flip, w[1] ^ flip, w[2] ^ flip, w[3] ^ flip};
        } else {
          unsigned char o[16];
#pragma unroll
          for (int l = 0; l < LV; ++l)
#pragma unroll
            for (int e = 0; e < PER; ++e) o[l * PER + e] = (unsigned char)quant_one<TS>(in[g][l].get(e), sc, zf, true);
          __builtin_memcpy(&ov, o, 16);
        }
        *reinterpret_cast<uintx4*>(reinterpret_cast<unsigned char*>(p.dst) + t * tile + ((int64_t)g * kThreads + threadIdx.x) * 16) = ov;
      }
    }
    done = ntiles * tile;
  }
  for (int64_t i = done + t0; i < p.n; i += stride) {
    const int c = (p.channels > 1) ? (int)((i / p.inner) % p.channels) : 0;
    const int q = quant_one<TS>(Store<TS>::ld(x + i), p.scale[c], p.zp ? (float)p.zp[c] : 0.f, p.dst_signed);
    if (p.dst_signed) reinterpret_cast<int8_t*>(p.dst)[i] = (int8_t)q;
    else if (p.dst_dt == DT_I8) reinterpret_cast<int8_t*>(p.dst)[i] = q_to_stored(q);
    else reinterpret_cast<uint8_t*>(p.dst)[i] = (uint8_t)q;
  }
}

// x = (q - zp) * scale
template <typename TD>
__global__ void __launch_bounds__(kThreads)
dequantize_kernel(QuantParams p) {
  TD* y = reinterpret_cast<TD*>(p.dst);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  auto level = [&](unsigned char raw) -> float {
    if (p.src_dt == DT_U8) return (float)raw;
    if (p.dst_signed) return (float)(int8_t)raw;
    return (float)q_from_stored((int8_t)raw);
  };
  int64_t done = 0;
  if (p.channels == 1 && (reinterpret_cast<uintptr_t>(p.src) & 7u) == 0 && (reinterpret_cast<uintptr_t>(p.dst) & 15u) == 0) {
    const float sc = p.scale[0], zf = p.zp ? (float)p.zp[0] : 0.f;
    const int64_t n8 = p.n / 8;
    for (int64_t i = t0; i < n8; i += stride) {
      const uintx2 rv = *reinterpret_cast<const uintx2*>(reinterpret_cast<const unsigned char*>(p.src) + i * 8);
      unsigned char r[8];
      __builtin_memcpy(r, &rv, 8);
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (level(r[e]) - zf) * sc;
      if constexpr (sizeof(TD) == 2) {
        Vec16<TD> o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o.set(e, v[e]);
        o.store(y + i * 8);
      } else {
        *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(y) + i * 8) = (floatx4){v[0], v[1], v[2], v[3]};
        *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(y) + i * 8 + 4) = (floatx4){v[4], v[5], v[6], v[7]};
      }
    }
    done = n8 * 8;
  }
  for (int64_t i = done + t0; i < p.n; i += stride) {
    const int c = (p.channels > 1) ? (int)((i / p.inner) % p.channels) : 0;
    const float zf = p.zp ? (float)p.zp[c] : 0.f;
    Store<TD>::st(y + i, (level(reinterpret_cast<const unsigned char*>(p.src)[i]) - zf) * p.scale[c]);
  }
}

__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Activation inside a group.  With 16-bit storage the result keeps 8 or 11
// significant bits, so the hardware exponential and reciprocal (1 ulp each)
// stand in for the library's exp and the IEEE division.
template <typename T>
__device__ __forceinline__ float fused_act(const float v, const ActKind act, const float a, const float b) {
  if constexpr (sizeof(T) == 2) {
    if (act == ACT_SIGMOID) return __builtin_amdgcn_rcpf(1.0f + __expf(-v));
    if (act == ACT_EXP) return __expf(v);
  }
  return apply_act(v, act, a, b);
}

// One launch for groups of unary / binary operators (see FusedGroup).  The
// registers of a program live in LDS, one column per thread, because the
// program addresses them at run time.  A thread runs every instruction for E
// consecutive points of its walk at once (register q, point e at
// regs[(q * E + e) * kThreads + thread]): the E loads of an instruction are in
// flight together and the decoding of the instruction is shared.
//
// Large groups are bound by memory and by their exponentials, small ones by the chain of
// instructions: about 0.33 us each when every one was fetched as it ran, with its operands'
// loads waiting one by one.  So the program and its views are copied to LDS first, the next
// instruction is read while the current one runs, the leading loads are issued four
// instructions at a time, and what the walk does not change is computed once per walk.
// (All of a program and its views is requested without a wait for their counts: the copy is on
// every workgroup's chain, four rounds of them in the launch below; 95 -> 91 us for all of the
// post-processing of 16 images.)
// Class scores of 16 images (13.6 M points, two sigmoids each, 116 MB): 74 us in three launches
// behind tiled copies of 47 us, 42 us in one without them.
// (FusedViewAt: offset and strides in bytes, so that base + offset is one address operand.)
template <typename I>
struct FusedViewAt { const char* base; I off; I st[4]; };

// base + offset in bytes, as an address in device memory (a pointer that comes out of LDS could
// point anywhere: its accesses would wait for those of LDS as well)
template <typename T, typename I>
__device__ __forceinline__ T* fused_at(const char* base, const I off) {
  typedef __attribute__((address_space(1))) char* GlobalPtr;
  return (T*)((GlobalPtr)(uintptr_t)base + off);
}

// One arithmetic instruction for N points (the result of N = 1 goes to all E).
template <typename T, int N, int E>
__device__ __forceinline__ void fused_op(const FusedInstr& in, float* r) {
  float x[N];
  const int a = in.a, b = in.b, dst = in.dst;
#pragma unroll
  for (int e = 0; e < N; ++e) x[e] = a < 0 ? in.fa : r[(a * E + e) * kThreads];   // a negative register number selects the immediate
  // (one decision per instruction, not one per point)
#define FUSED_EACH(EXPR) _Pragma("unroll") for (int e = 0; e < N; ++e) x[e] = EXPR; break
  if (in.op == FOP_UNARY) {
#define FUSED_ACT(K) case K: FUSED_EACH(fused_act<T>(x[e], K, in.fa, in.fb))
    switch ((ActKind)in.kind) {
      FUSED_ACT(ACT_SIGMOID);
      FUSED_ACT(ACT_EXP);
      FUSED_ACT(ACT_TANH);
      FUSED_ACT(ACT_RELU);
      FUSED_ACT(ACT_NEG);
      FUSED_ACT(ACT_GELU_ERF);
      FUSED_ACT(ACT_DIV_CONST);
      FUSED_ACT(ACT_SQRT);
      default:   // (the rarer ones, one point after the other: their code is there once)
#pragma unroll 1
        for (int e = 0; e < E; ++e)
          r[(dst * E + e) * kThreads] = fused_act<T>(r[(a * E + (e < N ? e : 0)) * kThreads], (ActKind)in.kind, in.fa, in.fb);
        return;
    }
#undef FUSED_ACT
  } else {
    float y[N];
#pragma unroll
    for (int e = 0; e < N; ++e) y[e] = b < 0 ? in.fa : r[(b * E + e) * kThreads];
    switch ((BinKind)in.kind) {
      case BIN_ADD: FUSED_EACH(x[e] + y[e]);
      case BIN_SUB: FUSED_EACH(x[e] - y[e]);
      case BIN_MUL: FUSED_EACH(x[e] * y[e]);
      default: FUSED_EACH(bin_op(x[e], y[e], (BinKind)in.kind));
    }
  }
#undef FUSED_EACH
#pragma unroll
  for (int e = 0; e < E; ++e) r[(dst * E + e) * kThreads] = x[e < N ? e : 0];
}

// a value that every lane read from the same place in LDS, in scalar registers
template <typename V>
__device__ __forceinline__ V fused_uniform(const V v) {
  int w[sizeof(V) / 4];
  __builtin_memcpy(w, &v, sizeof(V));
#pragma unroll
  for (int q = 0; q < (int)(sizeof(V) / 4); ++q) w[q] = __builtin_amdgcn_readfirstlane(w[q]);
  V o;
  __builtin_memcpy(&o, w, sizeof(V));
  return o;
}

// I is the type of the index arithmetic: 32-bit when the walk and every view fit
// (integer division and multiplication in 64 bits cost several times as much).
template <typename T, int E, typename I>
__device__ __forceinline__ void fused_walks(const FusedGroup* __restrict__ g, const FusedInstr* prog, const FusedViewAt<I>* views,
                                            float* r, const int64_t first, const int64_t stride) {
  const I d1 = (I)g->dims[1], d2 = (I)g->dims[2], d3 = (I)g->dims[3];
  const I walk = g->walk > 0 ? (I)g->walk : d2;
  const I pieces = (d2 + walk - 1) / walk;
  const int64_t total = g->dims[0] * g->dims[1] * (int64_t)pieces * g->dims[3];
  const bool whole = d2 % (I)E == 0 && walk % (I)E == 0;   // (no piece ends within E points)
  const int once_loads = g->n_once_loads, loads_end = once_loads + g->n_loads, once_end = loads_end + g->n_once, n_instr = g->n_instr;
  for (int64_t t64 = first; t64 < total; t64 += stride) {
    const I t = (I)t64;
    I q, q1, i0;
    if constexpr (sizeof(I) == 4) {
      q = fast_div(t, g->magic[0], g->shift[0]);
      q1 = fast_div(q, g->magic[1], g->shift[1]);
      i0 = fast_div(q1, g->magic[2], g->shift[2]);
    } else {
      q = t / d3;
      q1 = q / pieces;
      i0 = q1 / d1;
    }
    const I i3 = t - q * d3, piece = q - q1 * pieces, i1 = q1 - i0 * d1;
    const I i2_end = piece * walk + walk < d2 ? piece * walk + walk : d2;
    int k0 = 0;
    for (I i2 = piece * walk; i2 < i2_end; i2 += E) {
      const int live = i2_end - i2 < (I)E ? (int)(i2_end - i2) : E;
      auto at = [&](const FusedViewAt<I>& v) { return v.off + i0 * v.st[0] + i1 * v.st[1] + i2 * v.st[2] + i3 * v.st[3]; };
      auto load = [&](const int k, auto count) {   // `count` load instructions, all in flight
        constexpr int kCount = decltype(count)::value;
        float val[kCount][E];
        int dst[kCount];
#pragma unroll
        for (int u = 0; u < kCount; ++u) {
          const FusedInstr in = fused_uniform(prog[k + u]);
          const FusedViewAt<I> v = fused_uniform(views[in.a]);
          dst[u] = in.dst;
          const I from = at(v);
          if (whole) {
#pragma unroll
            for (int e = 0; e < E; ++e) val[u][e] = Store<T>::ld(fused_at<const T, I>(v.base, from + (I)e * v.st[2]));
          } else {
#pragma unroll
            for (int e = 0; e < E; ++e) val[u][e] = e < live ? Store<T>::ld(fused_at<const T, I>(v.base, from + (I)e * v.st[2])) : 0.f;
          }
        }
#pragma unroll
        for (int u = 0; u < kCount; ++u)
#pragma unroll
          for (int e = 0; e < E; ++e) r[(dst[u] * E + e) * kThreads] = val[u][e];
      };
      if constexpr (E <= 4) for (; k0 + 4 <= loads_end; k0 += 4) load(k0, std::integral_constant<int, 4>{});
      for (; k0 + 2 <= loads_end; k0 += 2) load(k0, std::integral_constant<int, 2>{});
      if (k0 < loads_end) load(k0, std::integral_constant<int, 1>{});
      k0 = once_loads;
      if (i2 == piece * walk)
        for (int k = loads_end; k < once_end; ++k) fused_op<T, 1, E>(fused_uniform(prog[k]), r);
      FusedInstr next = prog[once_end];
      for (int k = once_end; k < n_instr; ++k) {
        const FusedInstr in = fused_uniform(next);
        next = prog[k + 1];   // (one more than there are)
        if (in.op == FOP_LOAD) {
          load(k, std::integral_constant<int, 1>{});
        } else if (in.op == FOP_STORE) {
          const FusedViewAt<I> v = fused_uniform(views[in.dst]);
          const I from = at(v);
          float val[E];
#pragma unroll
          for (int e = 0; e < E; ++e) val[e] = r[(in.a * E + e) * kThreads];
          if (whole) {
#pragma unroll
            for (int e = 0; e < E; ++e) Store<T>::st(fused_at<T, I>(v.base, from + (I)e * v.st[2]), val[e]);
          } else {
#pragma unroll
            for (int e = 0; e < E; ++e)
              if (e < live) Store<T>::st(fused_at<T, I>(v.base, from + (I)e * v.st[2]), val[e]);
          }
        } else {
          fused_op<T, E, E>(in, r);
        }
      }
    }
  }
}

// U points of a chain, from point i2 of the walk on: their loads, the operators on the values in
// hand, their stores.
template <typename T, int U>
__device__ __forceinline__ void fused_chain_points(const FusedInstr* prog, const int first, const int last, const FusedViewAt<uint32_t>& in_view,
                                                   const FusedViewAt<uint32_t>& out_view, const uint32_t in_at, const uint32_t out_at,
                                                   const uint32_t i2, const bool live, const int once0, const float o0, const float o1,
                                                   const bool best_of, float& best, int& best_at) {
  float x[U];
#pragma unroll
  for (int u = 0; u < U; ++u) x[u] = live ? Store<T>::ld(fused_at<const T, uint32_t>(in_view.base, in_at + (i2 + u) * in_view.st[2])) : 0.f;
  for (int k = first; k < last; ++k) {
    const FusedInstr in = fused_uniform(prog[k]);
#define CHAIN_EACH(EXPR) _Pragma("unroll") for (int u = 0; u < U; ++u) x[u] = EXPR; break
    if (in.op == FOP_UNARY) {
      switch ((ActKind)in.kind) {
        case ACT_SIGMOID: CHAIN_EACH(fused_act<T>(x[u], ACT_SIGMOID, 0.f, 0.f));
        case ACT_EXP: CHAIN_EACH(fused_act<T>(x[u], ACT_EXP, 0.f, 0.f));
        case ACT_TANH: CHAIN_EACH(fused_act<T>(x[u], ACT_TANH, 0.f, 0.f));
        default: CHAIN_EACH(fused_act<T>(x[u], ACT_RELU, 0.f, 0.f));
      }
    } else {
      // (the other operand: an immediate or what the walk does not change; `pad[0]`: it is the left one)
      const int reg = in.pad[0] ? in.a : in.b;
      const float y = reg < 0 ? in.fa : reg == once0 ? o0 : o1;
      switch ((BinKind)in.kind) {
        case BIN_ADD: CHAIN_EACH(x[u] + y);
        case BIN_MUL: CHAIN_EACH(x[u] * y);
        default:
          if (in.pad[0]) { CHAIN_EACH(y - x[u]); }
          CHAIN_EACH(x[u] - y);
      }
    }
#undef CHAIN_EACH
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    T t;
    Store<T>::st(&t, x[u]);
    if (live) *fused_at<T, uint32_t>(out_view.base, out_at + (i2 + u) * out_view.st[2]) = t;
    if (best_of) {
      const float v = Store<T>::ld(&t);
      if (v > best || i2 + u == 0) { best = v; best_at = (int)i2 + u; }
    }
  }
}

// A chain (FusedGroup::chain): the values of a walk stay in vector registers, up to eight points at a
// time, and only the once section uses the registers in LDS, one point each.  64 consecutive points
// across the walks per wavefront; the four wavefronts of a workgroup share a walk between them, and
// workgroups do where there would be few.  A workgroup goes through several such groups of points, so
// that its copy of the program (3 us behind the start of the launch) is paid once and in one round.
// With best_of the class scores of a detector leave with each box's best one: the launch that read
// all of them again (14 us for 16 images) is gone.
// Class scores of 16 images (13.6 M points, 116 MB) beside the boxes: 45.0 -> 33.6 us, what is left
// being mostly the sigmoids (some 45 vector instructions a point); 20 points at a time 38.2, half the
// workgroups 39.4, the same number of turns for all of them 34.4.
template <typename T>
__device__ __forceinline__ void fused_chain(const FusedGroup* __restrict__ g, const FusedInstr* prog, const FusedViewAt<uint32_t>* views,
                                            float* r, const uint32_t block, const uint32_t blocks, float* __restrict__ best_ws,
                                            int32_t* __restrict__ at_ws) {
  __shared__ float s_best[4][64];
  __shared__ int s_at[4][64];
  const uint32_t d0 = (uint32_t)g->dims[0], d1 = (uint32_t)g->dims[1], d2 = (uint32_t)g->dims[2], d3 = (uint32_t)g->dims[3];
  const uint32_t cols = d0 * d1 * d3, walk = (uint32_t)g->walk, split = (uint32_t)g->chain;
  const int once_loads = g->n_once_loads, loads_end = once_loads + 1, once_end = loads_end + g->n_once, last = g->n_instr - 1;
  const bool best_of = g->best_of != 0;
  const int once0 = g->chain_once[0], once1 = g->chain_once[1];
  const FusedViewAt<uint32_t> vin = fused_uniform(views[prog[once_loads].a]), vout = fused_uniform(views[prog[last].dst]);
  const int lane = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t turns = (cols + 63) / 64 * split;
  for (uint32_t t = block; t < turns; t += blocks) {
    const uint32_t group = split == 1 ? t : t / split, piece = (split == 1 ? 0 : t - group * split) * 4 + part;
    const uint32_t c = group * 64 + lane, col = c < cols ? c : cols - 1;
    const bool live = c < cols;
    const uint32_t q = fast_div(col, g->magic[0], g->shift[0]), i3 = col - q * d3;
    const uint32_t i0 = fast_div(q, g->magic[2], g->shift[2]), i1 = q - i0 * d1;
    for (int k = 0; k < once_loads; ++k) {
      const FusedInstr in = fused_uniform(prog[k]);
      const FusedViewAt<uint32_t> v = fused_uniform(views[in.a]);
      r[in.dst * kThreads] = Store<T>::ld(fused_at<const T, uint32_t>(v.base, v.off + i0 * v.st[0] + i1 * v.st[1] + i3 * v.st[3]));
    }
    for (int k = loads_end; k < once_end; ++k) fused_op<T, 1, 1>(fused_uniform(prog[k]), r);
    const float o0 = r[once0 * kThreads], o1 = r[once1 * kThreads];
    const uint32_t in_at = vin.off + i0 * vin.st[0] + i1 * vin.st[1] + i3 * vin.st[3];
    const uint32_t out_at = vout.off + i0 * vout.st[0] + i1 * vout.st[1] + i3 * vout.st[3];
    const uint32_t from = piece * walk, end = from + walk < d2 ? from + walk : d2;
    float best = -INFINITY;
    int best_at = (int)(from < d2 ? from : 0);
    uint32_t i2 = from;
#define CHAIN_POINTS(U) fused_chain_points<T, U>(prog, once_end, last, vin, vout, in_at, out_at, i2, live, once0, o0, o1, best_of, best, best_at)
    for (; i2 + 8 <= end; i2 += 8) CHAIN_POINTS(8);
    if (i2 + 4 <= end) { CHAIN_POINTS(4); i2 += 4; }
    for (; i2 < end; ++i2) CHAIN_POINTS(1);
#undef CHAIN_POINTS
    if (best_of) {   // (uniform over the workgroup)
      s_best[part][lane] = best;
      s_at[part][lane] = best_at;
      __syncthreads();
      if (part == 0 && live) {
#pragma unroll
        for (int w = 1; w < 4; ++w)
          if (s_best[w][lane] > best) { best = s_best[w][lane]; best_at = s_at[w][lane]; }
        const int64_t to = g->best_off + i0 * g->best_st[0] + i1 * g->best_st[1] + i3 * g->best_st[2];
        best_ws[to] = best;
        at_ws[to] = best_at;
      }
      __syncthreads();
    }
  }
}

template <typename T, typename I>
__global__ void __launch_bounds__(kThreads) fused_eltwise_kernel(const FusedLaunch l) {
  extern __shared__ float fused_regs[];
  __shared__ uintx4 s_code[kFusedMaxInstr + 1];
  FusedInstr* s_prog = reinterpret_cast<FusedInstr*>(s_code);
  __shared__ FusedViewAt<I> s_view[kFusedMaxViews];
  int n = 0;
  while (n + 1 < l.n_groups && (int)blockIdx.x >= l.block0[n + 1]) ++n;
  const FusedGroup* __restrict__ g = l.group[n];
  // (all there is room for, whether it is used or not: without a wait for the counts)
  static_assert(kFusedMaxInstr <= kThreads && kFusedMaxViews <= kThreads, "an instruction and a view per thread");
  FusedInstr in = {};
  FusedView v = {};
  const void* base = nullptr;
  if (threadIdx.x < kFusedMaxInstr) in = g->prog[threadIdx.x];
  if (threadIdx.x < kFusedMaxViews) {
    v = g->view[threadIdx.x];
    const int at = l.view0[n] + (int)threadIdx.x;
    base = l.base[at < kFusedMaxBases ? at : kFusedMaxBases - 1];
  }
  if (threadIdx.x < kFusedMaxInstr) s_prog[threadIdx.x] = in;
  if (threadIdx.x < kFusedMaxViews) {
    constexpr I es = (I)sizeof(T);
    s_view[threadIdx.x] = FusedViewAt<I>{reinterpret_cast<const char*>(base), (I)v.off * es,
                                         {(I)v.st[0] * es, (I)v.st[1] * es, (I)v.st[2] * es, (I)v.st[3] * es}};
  }
  __syncthreads();
  float* r = fused_regs + threadIdx.x;
  if constexpr (sizeof(I) == 4) {
    if (g->chain > 0) {
      fused_chain<T>(g, s_prog, s_view, r, blockIdx.x - l.block0[n], l.block0[n + 1] - l.block0[n], l.best, l.best_at);
      return;
    }
  }
  const int64_t first = (int64_t)((int)blockIdx.x - l.block0[n]) * kThreads + threadIdx.x;
  const int64_t stride = (int64_t)(l.block0[n + 1] - l.block0[n]) * kThreads;
  if (g->points == 8) fused_walks<T, 8, I>(g, s_prog, s_view, r, first, stride);
  else if (g->points == 4) fused_walks<T, 4, I>(g, s_prog, s_view, r, first, stride);
  else if (g->points == 2) fused_walks<T, 2, I>(g, s_prog, s_view, r, first, stride);
  else fused_walks<T, 1, I>(g, s_prog, s_view, r, first, stride);
}

}  // namespace

#define FLOAT_DISPATCH(dt, EXPR)                         \
  switch (dt) {                                          \
    case DT_F32: { using T = float; EXPR; break; }       \
    case DT_F16: { using T = f16_t; EXPR; break; }       \
    case DT_BF16: { using T = bf16_t; EXPR; break; }     \
    default: return hipErrorInvalidValue;                \
  }

hipError_t launch_unary(const void* x, void* y, DType dt, int64_t n, ActKind act, float a, float b,
                        hipStream_t stream) {
  if (n <= 0) return n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!x || !y || !al16(x) || !al16(y)) return hipErrorInvalidValue;
  constexpr int U = 4;
  const int64_t tiles = (n / (16 / dtype_size(dt)) + kThreads * U - 1) / (kThreads * U);
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(tiles > 0 ? tiles : 1));
#define UNARY_CASE(K_)                                                                                  \
  case K_:                                                                                              \
    FLOAT_DISPATCH(dt, hipLaunchKernelGGL((unary_kernel<T, (int)K_, U>), grid, dim3(kThreads), 0, stream, \
                                          (const T*)x, (T*)y, n, act, a, b));                           \
    break;
  switch (act) {
    UNARY_CASE(ACT_RELU)
    UNARY_CASE(ACT_LEAKY)
    UNARY_CASE(ACT_CLAMP)
    UNARY_CASE(ACT_NEG)
    UNARY_CASE(ACT_SIGMOID)
    UNARY_CASE(ACT_TANH)
    UNARY_CASE(ACT_GELU_ERF)
    UNARY_CASE(ACT_GELU_TANH)
    UNARY_CASE(ACT_EXP)
    default:
      FLOAT_DISPATCH(dt, hipLaunchKernelGGL((unary_kernel<T, -1, U>), grid, dim3(kThreads), 0, stream, (const T*)x,
                                            (T*)y, n, act, a, b));
  }
#undef UNARY_CASE
  return hipGetLastError();
}

hipError_t launch_channel_affine(const void* x, void* y, DType dt, int64_t n, int64_t inner,
                                 int channels, const float* scale, const float* shift,
                                 hipStream_t stream) {
  if (n <= 0) return n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!x || !y || !scale || !shift || !al16(x) || !al16(y) || inner <= 0 || channels <= 0)
    return hipErrorInvalidValue;
  if (n % (inner * channels) != 0) return hipErrorInvalidValue;
  constexpr int U = 4;
  const int64_t tiles = (n / (16 / dtype_size(dt)) + kThreads * U - 1) / (kThreads * U);
  if (tiles > 0x7fffffff) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)(tiles > 0 ? tiles : 1);
  FLOAT_DISPATCH(dt, hipLaunchKernelGGL((channel_affine_kernel<T, U>), dim3(grid), dim3(kThreads), 0,
                                        stream, (const T*)x, (T*)y, n, inner, channels, scale, shift));
  return hipGetLastError();
}

hipError_t launch_channel_rows(const ChannelRowsParams& p_in, hipStream_t stream) {
  ChannelRowsParams p = p_in;
  const bool affine = p.scale != nullptr, has_r = p.r != nullptr;
  if (!p.x || !p.y || p.rows <= 0 || p.C <= 0 || p.xcs < p.C || p.ycs < p.C || (has_r && p.rcs < p.C) || (affine && !p.shift))
    return hipErrorInvalidValue;
  const int v = 16 / dtype_size(p.dt);
  const bool vec = p.C % v == 0 && p.xcs % v == 0 && p.ycs % v == 0 && al16(p.x) && al16(p.y) &&
                   (!has_r || (p.rcs % v == 0 && al16(p.r)));
  const int w = vec ? v : 1;
  if (p.rows * (p.C / w) >= (1ll << 31)) return hipErrorInvalidValue;
  div_magic(p.C / w, &p.cw_magic, &p.cw_shift);
  constexpr int U = 4;
  const dim3 grid((unsigned)((p.rows * (p.C / w) + kThreads * U - 1) / (kThreads * U)));
#define ROWS_GO(W_, A_, OP_, K_) hipLaunchKernelGGL((channel_rows_kernel<T, W_, A_, OP_, K_, U>), grid, dim3(kThreads), 0, stream, p)
#define ROWS_ACT(W_, A_, OP_)                                         \
  do {                                                                \
    if (p.act == ACT_NONE) ROWS_GO(W_, A_, OP_, (int)ACT_NONE);       \
    else if (p.act == ACT_RELU) ROWS_GO(W_, A_, OP_, (int)ACT_RELU);  \
    else if (p.act == ACT_LEAKY) ROWS_GO(W_, A_, OP_, (int)ACT_LEAKY); \
    else ROWS_GO(W_, A_, OP_, -1);                                    \
  } while (0)
#define ROWS_CASE(W_)                                                                            \
  do {                                                                                           \
    if (affine && !has_r) ROWS_ACT(W_, true, -2);                                                \
    else if (!affine && has_r && p.op == BIN_ADD) ROWS_ACT(W_, false, (int)BIN_ADD);             \
    else if (!affine && has_r) ROWS_GO(W_, false, -1, -1);                                       \
    else if (!affine) ROWS_ACT(W_, false, -2);                                                   \
    else ROWS_GO(W_, true, -1, -1);                                                              \
  } while (0)
  FLOAT_DISPATCH(p.dt, do { if (vec) ROWS_CASE(16 / (int)sizeof(T)); else ROWS_CASE(1); } while (0));
#undef ROWS_CASE
#undef ROWS_ACT
#undef ROWS_GO
  return hipGetLastError();
}

hipError_t launch_bn_fold(const float* mean, const float* var, const float* gamma,
                          const float* beta, float sgamma, float sbeta, float eps, int channels,
                          float* scale, float* shift, hipStream_t stream) {
  if (!mean || !var || !scale || !shift || channels <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(bn_fold_kernel, dim3((channels + 255) / 256), dim3(256), 0, stream, mean, var,
                     gamma, beta, sgamma, sbeta, eps, channels, scale, shift);
  return hipGetLastError();
}

hipError_t launch_binary(const BinaryParams& p, hipStream_t stream) {
  if (!p.a || !p.b || !p.y || p.rank < 1 || p.rank > 6) return hipErrorInvalidValue;
  int64_t n = 1;
  for (int d = 0; d < p.rank; ++d) {
    if (p.dims[d] <= 0) return hipErrorInvalidValue;
    n *= p.dims[d];
  }
  // contiguous strides of the output
  int64_t cs[6];
  {
    int64_t s = 1;
    for (int d = p.rank - 1; d >= 0; --d) { cs[d] = s; s *= p.dims[d]; }
  }
  auto is_full = [&](const int64_t* st) {
    for (int d = 0; d < p.rank; ++d)
      if (p.dims[d] != 1 && st[d] != cs[d]) return false;
    return true;
  };
  // operand indexed only by a trailing block of dims (contiguous there), 0 elsewhere
  auto rowvec_period = [&](const int64_t* st) -> int64_t {
    int d = p.rank - 1;
    int64_t period = 1;
    while (d >= 0 && (p.dims[d] == 1 || st[d] == cs[d])) { period *= p.dims[d]; --d; }
    for (; d >= 0; --d)
      if (p.dims[d] != 1 && st[d] != 0) return -1;
    return period;
  };
  const int grid = grid_for(n, kThreads * 8);
  if (p.dt == DT_I8) {
    if (!is_full(p.sa) || !is_full(p.sb) || !al16(p.a) || !al16(p.b) || !al16(p.y))
      return hipErrorInvalidValue;
    hipLaunchKernelGGL(binary_q8_kernel, dim3(grid_for(n, kThreads * 16)), dim3(kThreads), 0, stream, p, n);
    return hipGetLastError();
  }
  const bool aligned = al16(p.a) && al16(p.b) && al16(p.y);
  if (aligned && is_full(p.sa) && is_full(p.sb)) {
    constexpr int U = 4;
    const int64_t tiles = (n / (16 / dtype_size(p.dt)) + kThreads * U - 1) / (kThreads * U);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 fgrid((unsigned)(tiles > 0 ? tiles : 1));
#define BIN_FLAT(OP_, K_)                                                                                           \
  FLOAT_DISPATCH(p.dt, hipLaunchKernelGGL((binary_flat_kernel<T, OP_, K_, U>), fgrid, dim3(kThreads), 0, stream,     \
                                          (const T*)p.a, (const T*)p.b, (T*)p.y, n, p.op, p.act, p.act_a, p.act_b))
    if (p.op == BIN_ADD && p.act == ACT_NONE) { BIN_FLAT((int)BIN_ADD, (int)ACT_NONE); }
    else if (p.op == BIN_ADD && p.act == ACT_RELU) { BIN_FLAT((int)BIN_ADD, (int)ACT_RELU); }
    else if (p.op == BIN_MUL && p.act == ACT_NONE) { BIN_FLAT((int)BIN_MUL, (int)ACT_NONE); }
    else if (p.op == BIN_SUB && p.act == ACT_NONE) { BIN_FLAT((int)BIN_SUB, (int)ACT_NONE); }
    else { BIN_FLAT(-1, -1); }
#undef BIN_FLAT
    return hipGetLastError();
  }
  if (aligned && is_full(p.sa)) {
    const int64_t per = rowvec_period(p.sb);
    if (per > 0 && per < (1ll << 30)) {
      FLOAT_DISPATCH(p.dt, hipLaunchKernelGGL(binary_rowvec_kernel<T>, dim3(grid), dim3(kThreads), 0,
                                              stream, (const T*)p.a, (const T*)p.b, (T*)p.y, n, (int)per,
                                              false, p.op, p.act, p.act_a, p.act_b));
      return hipGetLastError();
    }
  }
  if (aligned && is_full(p.sb)) {
    const int64_t per = rowvec_period(p.sa);
    if (per > 0 && per < (1ll << 30)) {
      FLOAT_DISPATCH(p.dt, hipLaunchKernelGGL(binary_rowvec_kernel<T>, dim3(grid), dim3(kThreads), 0,
                                              stream, (const T*)p.b, (const T*)p.a, (T*)p.y, n, (int)per,
                                              true, p.op, p.act, p.act_a, p.act_b));
      return hipGetLastError();
    }
  }
  FLOAT_DISPATCH(p.dt, hipLaunchKernelGGL(binary_bcast_kernel<T>, dim3(grid_for(n, kThreads * 2)),
                                          dim3(kThreads), 0, stream, p, n));
  return hipGetLastError();
}

hipError_t launch_scalar_chain(const void* src, DType sdt, void* dst, DType ddt, int64_t n, const ScalarChain& s, hipStream_t stream) {
  if (!src || !dst || n <= 0 || s.n < 1 || s.n > kScalarChain) return hipErrorInvalidValue;
  const int grid = grid_for(n, kThreads * 4);
#define CHAIN_CASE(S_, D_, TS_, TD_) \
  if (sdt == S_ && ddt == D_) {      \
    hipLaunchKernelGGL((scalar_chain_kernel<TS_, TD_>), dim3(grid), dim3(kThreads), 0, stream, (const TS_*)src, (TD_*)dst, n, s); \
    return hipGetLastError();        \
  }
  CHAIN_CASE(DT_F32, DT_F32, float, float)
  CHAIN_CASE(DT_F32, DT_F16, float, f16_t)
  CHAIN_CASE(DT_F32, DT_BF16, float, bf16_t)
  CHAIN_CASE(DT_F16, DT_F16, f16_t, f16_t)
  CHAIN_CASE(DT_BF16, DT_BF16, bf16_t, bf16_t)
#undef CHAIN_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_cast(const void* src, DType sdt, void* dst, DType ddt, int64_t n, hipStream_t stream) {
  if (n <= 0) return n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!src || !dst) return hipErrorInvalidValue;
  const int grid = grid_for(n, kThreads * 4);
#define CAST_CASE(S_, D_, TS_, TD_, K_)                                                   \
  if (sdt == S_ && ddt == D_) {                                                           \
    hipLaunchKernelGGL((K_<TS_, TD_>), dim3(grid), dim3(kThreads), 0, stream, (const TS_*)src, \
                       (TD_*)dst, n);                                                     \
    return hipGetLastError();                                                             \
  }
  CAST_CASE(DT_F32, DT_F16, float, f16_t, cast_kernel)
  CAST_CASE(DT_F32, DT_BF16, float, bf16_t, cast_kernel)
  CAST_CASE(DT_F16, DT_F32, f16_t, float, cast_kernel)
  CAST_CASE(DT_BF16, DT_F32, bf16_t, float, cast_kernel)
  CAST_CASE(DT_F32, DT_F32, float, float, cast_kernel)
  CAST_CASE(DT_F16, DT_F16, f16_t, f16_t, cast_kernel)
  CAST_CASE(DT_BF16, DT_BF16, bf16_t, bf16_t, cast_kernel)
  CAST_CASE(DT_F16, DT_BF16, f16_t, bf16_t, cast_kernel)
  CAST_CASE(DT_BF16, DT_F16, bf16_t, f16_t, cast_kernel)
#define CAST_INT_CASE(S_, D_, TS_, TD_, B_)                                                  \
  if (sdt == S_ && ddt == D_) {                                                              \
    hipLaunchKernelGGL((cast_int_kernel<TS_, TD_, B_>), dim3(grid), dim3(kThreads), 0, stream, \
                       (const TS_*)src, (TD_*)dst, n);                                       \
    return hipGetLastError();                                                                \
  }
  // every source type to every integer type and bool ...
#define CAST_TO_INTS(S_, TS_)                        \
  CAST_INT_CASE(S_, DT_I8, TS_, int8_t, false)       \
  CAST_INT_CASE(S_, DT_U8, TS_, uint8_t, false)      \
  CAST_INT_CASE(S_, DT_I32, TS_, int32_t, false)     \
  CAST_INT_CASE(S_, DT_I64, TS_, int64_t, false)     \
  CAST_INT_CASE(S_, DT_BOOL, TS_, uint8_t, true)
  CAST_TO_INTS(DT_F32, float)
  CAST_TO_INTS(DT_F16, f16_t)
  CAST_TO_INTS(DT_BF16, bf16_t)
  CAST_TO_INTS(DT_I8, int8_t)
  CAST_TO_INTS(DT_U8, uint8_t)
  CAST_TO_INTS(DT_I32, int32_t)
  CAST_TO_INTS(DT_I64, int64_t)
  CAST_TO_INTS(DT_BOOL, uint8_t)
  // ... and every integer type and bool to every floating-point type
#define CAST_TO_FLOATS(S_, TS_)                      \
  CAST_INT_CASE(S_, DT_F32, TS_, float, false)       \
  CAST_INT_CASE(S_, DT_F16, TS_, f16_t, false)       \
  CAST_INT_CASE(S_, DT_BF16, TS_, bf16_t, false)
  CAST_TO_FLOATS(DT_I8, int8_t)
  CAST_TO_FLOATS(DT_U8, uint8_t)
  CAST_TO_FLOATS(DT_I32, int32_t)
  CAST_TO_FLOATS(DT_I64, int64_t)
  CAST_TO_FLOATS(DT_BOOL, uint8_t)
#undef CAST_TO_FLOATS
#undef CAST_TO_INTS
#undef CAST_INT_CASE
#undef CAST_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_quantize(const QuantParams& p, hipStream_t stream) {
  if (p.n <= 0) return p.n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!p.src || !p.dst || !p.scale || p.channels <= 0 || p.inner <= 0) return hipErrorInvalidValue;
  if (p.dst_dt != DT_U8 && p.dst_dt != DT_I8) return hipErrorInvalidValue;
  const int grid = grid_for(p.n, kThreads * 16);
  FLOAT_DISPATCH(p.src_dt, hipLaunchKernelGGL(quantize_kernel<T>, dim3(grid), dim3(kThreads), 0, stream, p));
  return hipGetLastError();
}

hipError_t launch_dequantize(const QuantParams& p, hipStream_t stream) {
  if (p.n <= 0) return p.n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!p.src || !p.dst || !p.scale || p.channels <= 0 || p.inner <= 0) return hipErrorInvalidValue;
  if (p.src_dt != DT_U8 && p.src_dt != DT_I8) return hipErrorInvalidValue;
  const int grid = grid_for(p.n, kThreads * 16);
  FLOAT_DISPATCH(p.dst_dt, hipLaunchKernelGGL(dequantize_kernel<T>, dim3(grid), dim3(kThreads), 0, stream, p));
  return hipGetLastError();
}

hipError_t launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t stream) {
  if (n <= 0) return n == 0 ? hipSuccess : hipErrorInvalidValue;
  if (!p) return hipErrorInvalidValue;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, p, n, v);
  return hipGetLastError();
}

constexpr int kChainBlocks = 256 * 6;   // workgroups of a chain

bool fused_prepare(FusedGroup* g, int* blocks, size_t* lds_bytes, bool* wide) {
  if (g->n_instr <= 0 || g->n_instr > kFusedMaxInstr || g->n_views < 0 || g->n_views > kFusedMaxViews) return false;
  if (g->n_once_loads < 0 || g->n_loads < 0 || g->n_once < 0) return false;
  const int loads_end = g->n_once_loads + g->n_loads, once_end = loads_end + g->n_once;
  if (once_end > g->n_instr) return false;
  int64_t threads = 1;
  for (int i = 0; i < 4; ++i) {
    if (g->dims[i] <= 0) return false;
    if (i != 2) threads *= g->dims[i];
  }
  if (g->walk < 0) return false;
  const int64_t walk = g->walk > 0 ? g->walk : g->dims[2];
  threads *= (g->dims[2] + walk - 1) / walk;
  int n_regs = 1;
  for (int k = 0; k < g->n_instr; ++k) {
    const FusedInstr& in = g->prog[k];
    if (in.op > FOP_STORE) return false;
    // (each section holds what the kernel takes it for)
    if (k < loads_end && in.op != FOP_LOAD) return false;
    if (k >= loads_end && k < once_end && in.op != FOP_UNARY && in.op != FOP_BINARY) return false;
    const bool is_store = in.op == FOP_STORE, is_load = in.op == FOP_LOAD, is_bin = in.op == FOP_BINARY;
    const int view = is_store ? in.dst : in.a;
    if ((is_store || is_load) && (view < 0 || view >= g->n_views)) return false;
    if (!is_store && (in.dst < 0 || in.dst >= kFusedMaxRegs)) return false;
    if (!is_load && (in.a >= kFusedMaxRegs || (in.a < 0 && !is_bin))) return false;
    if (is_bin && (in.b >= kFusedMaxRegs || (in.a < 0 && in.b < 0))) return false;
    if (!is_store && in.dst + 1 > n_regs) n_regs = in.dst + 1;
  }
  // A chain: behind the once section one load, operators on the value in hand (the other operand: an
  // immediate or one of at most two results of the once section), one store.  Walks of fewer than 16
  // points and launches of fewer than two wavefronts of neighbouring points stay on the general path.
  const int64_t cols = g->dims[0] * g->dims[1] * g->dims[3];
  bool chain = g->n_loads == 1 && g->n_instr > once_end && g->prog[g->n_instr - 1].op == FOP_STORE && g->dims[2] >= 16 && cols >= 128;
  if (chain) {
    unsigned once_regs = 0;
    for (int k = 0; k < once_end; ++k)
      if (k != g->n_once_loads) once_regs |= 1u << g->prog[k].dst;
    int used = 0, once[2] = {0, 0}, value = g->prog[g->n_once_loads].dst;
    for (int k = once_end; k + 1 < g->n_instr && chain; ++k) {
      FusedInstr& in = g->prog[k];
      if (in.op == FOP_UNARY) {
        chain = in.a == value && (in.kind == ACT_SIGMOID || in.kind == ACT_EXP || in.kind == ACT_TANH || in.kind == ACT_RELU);
      } else if (in.op == FOP_BINARY) {
        const bool right = in.b == value;
        const int other = right ? in.a : in.b;
        chain = (in.a == value) != right && (in.kind == BIN_ADD || in.kind == BIN_SUB || in.kind == BIN_MUL);
        if (chain && other >= 0 && !(used > 0 && once[0] == other) && !(used > 1 && once[1] == other)) {
          chain = (once_regs >> other & 1u) != 0 && used < 2;
          if (chain) once[used++] = other;
        }
        in.pad[0] = right ? 1 : 0;
      } else {
        chain = false;
      }
      value = in.dst;
      chain = chain && (once_regs >> value & 1u) == 0;
    }
    chain = chain && g->prog[g->n_instr - 1].a == value;
    g->chain_once[0] = once[0];
    g->chain_once[1] = used > 1 ? once[1] : once[0];
  }
  // points of the walk per instruction: as many as 32 KiB of LDS registers allow
  g->points = (walk >= 8 && n_regs * 8 <= 32) ? 8 : (walk >= 4 && n_regs * 4 <= 32) ? 4 : ((walk >= 2 && n_regs * 2 <= 32) ? 2 : 1);
  *lds_bytes = (size_t)n_regs * g->points * kThreads * sizeof(float);
  *blocks = grid_for(threads, kThreads, 256 * 8);   // (a workgroup spends 3 us on its copy of the program)
  // 32-bit index arithmetic when the thread count and every view's furthest element fit
  bool small = threads < ((int64_t)1 << 31);
  for (int v = 0; v < g->n_views && small; ++v) {
    int64_t far = g->view[v].off;
    if (far < 0) small = false;
    for (int q = 0; q < 4 && small; ++q) {
      if (g->view[v].st[q] < 0) small = false;
      else far += (g->dims[q] - 1 + (q == 2 ? g->points : 0)) * g->view[v].st[q];
    }
    if (far >= ((int64_t)1 << 29)) small = false;   // (bytes)
  }
  *wide = !small;
  g->chain = 0;
  if (chain && small) {
    // a workgroup's four wavefronts deal a walk between them, several workgroups where there are few
    const int64_t groups = (cols + 63) / 64;
    int64_t split = (1024 + groups - 1) / groups;
    if (split > g->dims[2] / 16) split = g->dims[2] / 16;
    if (g->best_of) split = 1;
    g->chain = (int)split;
    g->walk = ((g->dims[2] + 4 * split - 1) / (4 * split) + 3) / 4 * 4;
    g->points = 1;
    *lds_bytes = (size_t)n_regs * kThreads * sizeof(float);
    *blocks = (int)(groups * split < kChainBlocks ? groups * split : kChainBlocks);
  }
  const int64_t per = g->walk > 0 ? g->walk : g->dims[2];
  for (int v : {0, 1, 2}) {   // (32-bit walks: divisors of the thread number and what is left of it)
    const int64_t d = v == 0 ? g->dims[3] : v == 1 ? (g->dims[2] + per - 1) / per : g->dims[1];
    if (small) div_magic((int)d, &g->magic[v], &g->shift[v]);
  }
  return true;
}

hipError_t launch_fused_eltwise(const FusedLaunch& l, hipStream_t stream) {
  if (l.n_groups < 1 || l.n_groups > kFusedMaxGroups || l.view0[l.n_groups] > kFusedMaxBases) return hipErrorInvalidValue;
  for (int k = 0; k < l.n_groups; ++k)
    if (l.group[k] == nullptr || l.block0[k + 1] <= l.block0[k] || l.view0[k + 1] < l.view0[k]) return hipErrorInvalidValue;
  for (int k = 0; k < l.view0[l.n_groups]; ++k)
    if (l.base[k] == nullptr) return hipErrorInvalidValue;
  if (l.best != nullptr && (l.wide || l.best_at == nullptr)) return hipErrorInvalidValue;   // (only chains leave them)
  const dim3 grid((unsigned)l.block0[l.n_groups]);
  if (l.wide) { FLOAT_DISPATCH(l.dt, hipLaunchKernelGGL((fused_eltwise_kernel<T, int64_t>), grid, dim3(kThreads), l.lds_bytes, stream, l)); }
  else { FLOAT_DISPATCH(l.dt, hipLaunchKernelGGL((fused_eltwise_kernel<T, uint32_t>), grid, dim3(kThreads), l.lds_bytes, stream, l)); }
  return hipGetLastError();
}

}  // namespace ohip
