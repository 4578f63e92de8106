// Batched non-maximum suppression for gfx950: one launch over all boxes for the
// class reduction, then one workgroup per image.
//
// Phase 1  every box competes with its best class score (first maximum over
//          the class axis); boxes with score > score_thr become candidates.
//          scores are [C][B] per image, so for a fixed class consecutive lanes
//          read consecutive boxes.  The reduction over the classes reads the
//          whole score tensor and runs chip-wide; it leaves the decisions as
//          words of 64, of which the per-image workgroup makes its list.
// Phase 2  candidates are ordered by (score descending, box index ascending)
//          with a bitonic sort of 64-bit keys.
// Phase 3  greedy suppression in sorted order: an unsuppressed candidate is
//          emitted and the later candidates whose IoU with it is >= iou_thr are
//          marked.  A suppressed candidate never suppresses others, so the
//          result equals the sequential "compare with every kept box" rule.
//
// Up to 8192 candidates per image (the usual case by far) phases 2 and 3 keep
// everything on the compute unit: a thread holds its (up to eight) keys in
// registers, compare-exchange steps between lanes of a wavefront are lane
// shuffles, only steps between wavefronts go through LDS.  Phase 3 takes 64
// candidates at a time: the wavefronts share the 64 x 64 overlap tests (one
// ballot makes a row), every wavefront then resolves the greedy order of the
// block by itself on 64-bit masks, and the boxes kept are tested against all
// later candidates at once: two barriers per 64 candidates, where one per kept
// box (a chain of LDS reads, a test and a barrier of 16 wavefronts, 0.8 us)
// made 16 images of about 400 candidates take 91 us; now 17 us.  Longer
// lists are sorted and walked in the workspace.
//
// IoU uses the same fp32 operation order as the CPU formulation (corner boxes
// normalised with min/max, zero when either area is <= 0).  Boxes and scores
// are read in their storage type (fp32 / fp16 / bf16); the conversion to fp32 is
// exact.
#include "device_utils.h"

namespace ohip {
namespace {

constexpr int kNmsThreads = 1024;

__host__ __device__ inline int64_t next_pow2(int64_t v) {
  int64_t p = 1;
  while (p < v) p <<= 1;
  return p;
}

struct Box4 { float y1, x1, y2, x2; };

template <typename TB>
__device__ __forceinline__ Box4 norm_box(const TB* b) {
  const float b0 = Store<TB>::ld(b), b1 = Store<TB>::ld(b + 1), b2 = Store<TB>::ld(b + 2), b3 = Store<TB>::ld(b + 3);
  Box4 r;
  r.y1 = fminf(b0, b2);
  r.x1 = fminf(b1, b3);
  r.y2 = fmaxf(b0, b2);
  r.x2 = fmaxf(b1, b3);
  return r;
}

__device__ __forceinline__ float box_area(const Box4& a) { return (a.y2 - a.y1) * (a.x2 - a.x1); }

__device__ __forceinline__ float iou_of(const Box4& a, const float area_a, const Box4& b, const float area_b) {
  if (area_a <= 0.f || area_b <= 0.f) return 0.f;
  const float ih = fmaxf(fminf(a.y2, b.y2) - fmaxf(a.y1, b.y1), 0.f);
  const float iw = fmaxf(fminf(a.x2, b.x2) - fmaxf(a.x1, b.x1), 0.f);
  const float inter = ih * iw;
  return inter / (area_a + area_b - inter);
}

// min / max of values that came out of norm_box (no signalling NaN among them, so the
// canonicalising instruction that fminf / fmaxf would add to every operand has nothing to do);
// the first operand is the same in all lanes
__device__ __forceinline__ float min_of(const float uniform, const float v) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "s"(uniform), "v"(v));
  return r;
}
__device__ __forceinline__ float max_of(const float uniform, const float v) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "s"(uniform), "v"(v));
  return r;
}

// The lanes whose box b has iou_of(...) >= thr with box a (the same in all lanes), of those in `live`.
// No division in all but the closest cases: the quotient's rounding error is far below the margin
// of 1e-5, so outside it the products decide alike (not for tiny thresholds and areas, and NaN).
// Symmetric in the two boxes, like iou_of.
__device__ __forceinline__ unsigned long long overlaps(const Box4& a, const float area_a, const Box4& b, const float area_b,
                                                       const float thr, const unsigned long long live) {
  const float ih = fmaxf(min_of(a.y2, b.y2) - max_of(a.y1, b.y1), 0.f);
  const float iw = fmaxf(min_of(a.x2, b.x2) - max_of(a.x1, b.x1), 0.f);
  const float inter = ih * iw, t = thr * (area_a + area_b - inter);
  unsigned long long hit = __ballot(inter > t * 1.00001f);
  const unsigned long long below = __ballot(inter < t * 0.99999f);
  const unsigned long long known = __ballot(fminf(fminf(area_a, area_b), t) > 1e-30f) & (hit | below);
  hit &= live;
  if ((live & ~known) != 0 || !(thr > 1e-6f)) hit = __ballot(iou_of(a, area_a, b, area_b) >= thr) & live;
  return hit;
}

// best[n][b] = max over classes (first maximum), cls[n][b] = its class
// A workgroup takes 64 boxes; its four wavefronts share the classes (a quarter each, so that a
// single image keeps more than a handful of loads in flight), and the first combines them in
// class order.  Its 64 decisions leave as one word.
template <typename TS>
__global__ void __launch_bounds__(256)
nms_best_class_kernel(const TS* __restrict__ scores, int C, int B, float score_thr, float* __restrict__ best_ws,
                      int32_t* __restrict__ cls_ws, unsigned long long* __restrict__ mask_ws) {
  __shared__ float s_best[4][64];
  __shared__ int s_cls[4][64];
  const int n = blockIdx.y;
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int b = blockIdx.x * 64 + lane;
  const int per = (C + 3) / 4, end = (part + 1) * per < C ? (part + 1) * per : C;
  if (b < B) {
    const TS* sc = scores + (int64_t)n * C * B + b;
    int c = part * per;
    // (the walk starts with the first class as it is, a NaN included; the other parts
    //  start below everything)
    float best = -INFINITY;
    int bc = c;
    if (part == 0) best = Store<TS>::ld(sc + (int64_t)c++ * B);
    for (; c + 8 <= end; c += 8) {   // eight loads in flight; the comparisons keep the class order
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = Store<TS>::ld(sc + (int64_t)(c + u) * B);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (v[u] > best) { best = v[u]; bc = c + u; }
    }
    for (; c < end; ++c) {
      const float v = Store<TS>::ld(sc + (int64_t)c * B);
      if (v > best) { best = v; bc = c; }
    }
    s_best[part][lane] = best;
    s_cls[part][lane] = bc;
  }
  __syncthreads();
  if (part != 0) return;
  float best = s_best[0][lane];
  int bc = s_cls[0][lane];
#pragma unroll
  for (int q = 1; q < 4; ++q)
    if (s_best[q][lane] > best) { best = s_best[q][lane]; bc = s_cls[q][lane]; }
  const unsigned long long mask = __ballot(b < B && best > score_thr);
  if (lane == 0) mask_ws[(int64_t)n * gridDim.x + blockIdx.x] = mask;
  if (b >= B) return;
  best_ws[(int64_t)n * B + b] = best;
  cls_ws[(int64_t)n * B + b] = bc;
}

// One compare-exchange of the bitonic network seen from element i: `mine` stays or
// is replaced by `other` (the value of element i ^ j).
__device__ __forceinline__ unsigned long long bitonic_pick(const unsigned long long mine, const unsigned long long other,
                                                           const int i, const int j, const int k) {
  const bool lower = (i & j) == 0, up = (i & k) == 0;
  return ((mine < other) == (lower == up)) ? mine : other;
}

// the value of lane ^ J (J a power of two, within 64 lanes)
template <int J>
__device__ __forceinline__ unsigned long long lane_xor(const unsigned long long v) {
  int lo = (int)(unsigned)v, hi = (int)(unsigned)(v >> 32);
  if constexpr (J <= 2) {          // quad permutation: no LDS crossbar
    constexpr int kPerm = J == 1 ? 0xB1 : 0x4E;
    lo = __builtin_amdgcn_mov_dpp(lo, kPerm, 0xf, 0xf, true);
    hi = __builtin_amdgcn_mov_dpp(hi, kPerm, 0xf, 0xf, true);
  } else if constexpr (J < 32) {   // swizzle of 32 lanes: no address to make
    lo = __builtin_amdgcn_ds_swizzle(lo, (J << 10) | 0x1f);
    hi = __builtin_amdgcn_ds_swizzle(hi, (J << 10) | 0x1f);
  } else {
    lo = __shfl_xor(lo, J, 64);
    hi = __shfl_xor(hi, J, 64);
  }
  return ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
}

constexpr int kNmsPerThread = 8;   // candidates a thread holds at most when the list stays on the compute unit

template <int NPT, int J>
__device__ __forceinline__ void bitonic_lanes(unsigned long long* e, const int tid, const int R, const int k) {
  if (k > J) {
#pragma unroll
    for (int m = 0; m < NPT; ++m)
      if (NPT == 1 || m < R) e[m] = bitonic_pick(e[m], lane_xor<J>(e[m]), tid + m * kNmsThreads, J, k);
  }
  if constexpr (J > 1) bitonic_lanes<NPT, J / 2>(e, tid, R, k);
}

// Phases 2 and 3 for a list of at most lds_slots candidates (M of them, P = next
// power of two), whose keys phase 1 left in `lds` [0, M).  NPT = 1: P <= kNmsThreads (the code
// for several keys per thread made the sort of 512 keys take 18 us; this takes 4).
template <typename TB, int NPT>
__device__ __forceinline__ void nms_on_cu(const TB* __restrict__ bx, const int32_t* __restrict__ cls, int32_t* __restrict__ o,
                                          unsigned long long* lds, const int n, const int M, const int P,
                                          const int max_out, const float iou_thr) {
  const int tid = threadIdx.x;
  constexpr int kWaves = kNmsThreads / 64;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R = NPT > 1 ? P / kNmsThreads : 1;   // elements per thread: i = tid + m * kNmsThreads
  const bool sorts = wave * 64 < P;              // (a wavefront with keys to sort; uniform)
  unsigned long long e[NPT];
#pragma unroll
  for (int m = 0; m < NPT; ++m) {
    const int i = tid + m * kNmsThreads;
    e[m] = (m < R && i < M) ? lds[i] : ~0ull;
  }
  __syncthreads();   // the keys are in registers: LDS becomes two exchange buffers of P keys

  int xsel = 0;
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j >= 64; j >>= 1) {
      if (j >= kNmsThreads) {   // both elements in this thread
        if constexpr (NPT > 1) {
#pragma unroll
          for (int db = 0; db < 3; ++db) {
            if ((j / kNmsThreads) != (1 << db)) continue;
#pragma unroll
            for (int m = 0; m < NPT; ++m) {
              if ((m & (1 << db)) != 0 || m >= R) continue;
              const int i = tid + m * kNmsThreads;
              const unsigned long long a = e[m], b = e[m | (1 << db)];
              e[m] = bitonic_pick(a, b, i, j, k);
              e[m | (1 << db)] = bitonic_pick(b, a, i | j, j, k);
            }
          }
        }
      } else {                  // the other element is in another wavefront: through LDS
        unsigned long long* x = lds + xsel * P;
        xsel ^= 1;   // the buffers alternate, so one barrier per step is enough
        if (sorts) {
#pragma unroll
          for (int m = 0; m < NPT; ++m)
            if (m < R && tid + m * kNmsThreads < P) x[tid + m * kNmsThreads] = e[m];
        }
        __syncthreads();
        if (sorts) {
#pragma unroll
          for (int m = 0; m < NPT; ++m) {
            const int i = tid + m * kNmsThreads;
            if (m < R && i < P) e[m] = bitonic_pick(e[m], x[i ^ j], i, j, k);
          }
        }
      }
    }
    if (sorts) bitonic_lanes<NPT, 32>(e, tid, R, k);   // the other element is in another lane of this wavefront
  }
  __syncthreads();   // every exchange has been read: LDS becomes the candidates' boxes and flags

  Box4* lbox = reinterpret_cast<Box4*>(lds);
  unsigned char* lsup = reinterpret_cast<unsigned char*>(lbox + P);
  __shared__ unsigned long long s_row[64];
  int mbi[NPT], mcls[NPT], mrow[NPT];
#pragma unroll
  for (int m = 0; m < NPT; ++m) {
    const int i = tid + m * kNmsThreads;
    mbi[m] = 0;
    mcls[m] = 0;
    mrow[m] = -1;
    if (m < R && i < M) {
      mbi[m] = (int)(e[m] & 0xffffffffu);
      lbox[i] = norm_box(bx + (int64_t)mbi[m] * 4);
      mcls[m] = cls[mbi[m]];
      lsup[i] = 0;
    }
  }
  __syncthreads();

  int kept = 0;   // every wavefront counts the kept boxes itself
  for (int base = 0; base < M && kept < max_out; base += 64) {
    const int mine = base + lane;
    const unsigned long long open = __ballot(mine < M && lsup[mine < M ? mine : 0] == 0);   // the block's live candidates
    if (open == 0) continue;   // (uniform over the workgroup: the flags are behind a barrier)
    // every lane holds a box of the block; a box all lanes test against comes by lane broadcasts
    const Box4 bj = lbox[mine < M ? mine : 0];
    const float area_j = box_area(bj);
    auto of_lane = [&](const float v, const int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i)); };
    auto box_of = [&](const int i) { return Box4{of_lane(bj.y1, i), of_lane(bj.x1, i), of_lane(bj.y2, i), of_lane(bj.x2, i)}; };
    // row i: the candidates of the block that overlap candidate i
#pragma unroll 1
    for (int q = 0; q < 64 / kWaves; ++q) {
      const int i = wave * (64 / kWaves) + q;
      unsigned long long row = 0;
      if ((open >> i) & 1ull) row = overlaps(box_of(i), of_lane(area_j, i), bj, area_j, iou_thr, open);
      if (lane == 0) s_row[i] = row;
    }
    __syncthreads();
    // The greedy order within the block: a candidate stays once every earlier one that overlaps it
    // is known to go, and goes once one is known to stay; as many rounds as the longest such chain.
    const unsigned long long before = s_row[lane] & ((1ull << lane) - 1);
    unsigned long long keep = 0, undecided = open;
    while (undecided != 0) {
      const bool here = ((undecided >> lane) & 1ull) != 0;
      const unsigned long long stay = __ballot(here && (before & (undecided | keep)) == 0);
      const unsigned long long go = __ballot(here && (before & keep) != 0);
      keep |= stay;
      undecided &= ~(stay | go);
    }
    if (__popcll(keep) > max_out - kept) {   // (the first ones of them)
      const unsigned long long first = __ballot(__popcll(keep & ((1ull << lane) - 1)) < max_out - kept);
      keep &= first;
    }
    if (wave == (base & (kNmsThreads - 1)) / 64 && ((keep >> lane) & 1ull)) {   // the owners note the output rows
      const int row = kept + __popcll(keep & ((1ull << lane) - 1));
#pragma unroll
      for (int m = 0; m < NPT; ++m)
        if (m == base / kNmsThreads) mrow[m] = row;
    }
    kept += __popcll(keep);
    if (kept >= max_out) break;
    // The boxes kept against the candidates behind the block: 64 candidates per wavefront, and
    // while that leaves wavefronts over, 2, 4, .. of them share the kept boxes of one group.
    const int groups = (M - base - 1) / 64;
    int parts = 1;
    unsigned long long share = ~0ull;   // every `parts`-th box of the block
    if (groups * 16 <= kWaves) { parts = 16; share = 0x0001000100010001ull; }
    else if (groups * 8 <= kWaves) { parts = 8; share = 0x0101010101010101ull; }
    else if (groups * 4 <= kWaves) { parts = 4; share = 0x1111111111111111ull; }
    else if (groups * 2 <= kWaves) { parts = 2; share = 0x5555555555555555ull; }
    const unsigned long long against = keep & (share << (wave % parts));
    if (against != 0) {
      for (int g = wave / parts; g < groups; g += kWaves / parts) {
        const int j = base + 64 * (g + 1) + lane;
        const Box4 b = lbox[j < M ? j : 0];
        const float area_b = box_area(b);
        unsigned long long live = __ballot(j < M && lsup[j < M ? j : 0] == 0), gone = 0;
        for (unsigned long long k = against; k != 0 && live != 0; k &= k - 1) {
          const int i = __builtin_amdgcn_readfirstlane(__ffsll(k) - 1);
          const unsigned long long hit = overlaps(box_of(i), of_lane(area_j, i), b, area_b, iou_thr, live);
          gone |= hit;
          live &= ~hit;
        }
        if ((gone >> lane) & 1ull) lsup[j] = 1;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < NPT; ++m) {
    if (mrow[m] >= 0) {
      o[mrow[m] * 3 + 0] = n;
      o[mrow[m] * 3 + 1] = mcls[m];
      o[mrow[m] * 3 + 2] = mbi[m];
    }
  }
}

template <typename TB>
__global__ void __launch_bounds__(kNmsThreads)
nms_kernel(const TB* __restrict__ boxes, const float* __restrict__ best_ws, int B,
           int max_out, float iou_thr, float score_thr, const unsigned long long* __restrict__ mask_ws, int32_t* __restrict__ out,
           unsigned long long* keys_ws, const int32_t* cls_ws, unsigned char* sup_ws, int64_t bpad,
           int lds_slots, int image_base) {
  const int n = blockIdx.x;
  const int tid = threadIdx.x;
  const TB* bx = boxes + (int64_t)n * B * 4;
  const float* bestv = best_ws + (int64_t)n * B;
  unsigned long long* keys = keys_ws + (int64_t)n * bpad;
  const int32_t* cls = cls_ws + (int64_t)n * B;
  unsigned char* sup = sup_ws + (int64_t)n * bpad;
  int32_t* o = out + (int64_t)n * max_out * 3;
  extern __shared__ unsigned long long lds_keys[];

  __shared__ int s_count;
  if (tid == 0) s_count = 0;
  for (int i = tid; i < max_out * 3; i += kNmsThreads) o[i] = -1;
  __syncthreads();

  // ---- phase 1 (second half): the boxes above the threshold, in no order, and their keys ----
  auto key_of = [](const float score, const unsigned b) {
    unsigned w = __float_as_uint(score);
    w = (w & 0x80000000u) ? ~w : (w | 0x80000000u);  // ascending in w == ascending in value
    return ((unsigned long long)(~w) << 32) | b;     // score desc, then box asc
  };
  if (mask_ws == nullptr) {
    // no words of decisions: the scores themselves, up to 24 per thread in flight (all boxes of a
    // 608 x 608 image at once; eight at a time took 3 us more there), and the keys at once
    constexpr int kAhead = 24;
    for (int b0 = 0; b0 < B; b0 += kAhead * kNmsThreads) {
      float v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int b = b0 + u * kNmsThreads + tid;
        if (b0 + u * kNmsThreads < B) v[u] = bestv[b < B ? b : B - 1];
      }
      // (one place in the list per wavefront for all of them: an atomic each took 3 us)
      unsigned long long mask[kAhead];
      int mine = 0;
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        mask[u] = 0;
        if (b0 + u * kNmsThreads < B) mask[u] = __ballot(b0 + u * kNmsThreads + tid < B && v[u] > score_thr);
        mine += __popcll(mask[u]);
      }
      if (mine == 0) continue;
      int slot = 0;
      if ((tid & 63) == 0) slot = atomicAdd(&s_count, mine);
      slot = __builtin_amdgcn_readfirstlane(slot);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int at = slot + __popcll(mask[u] & ((1ull << (tid & 63)) - 1));
        if ((mask[u] >> (tid & 63)) & 1ull) (at < lds_slots ? lds_keys : keys)[at] = key_of(v[u], (unsigned)(b0 + u * kNmsThreads + tid));
        slot += __popcll(mask[u]);
      }
    }
  } else {
    const int words = (B + 63) / 64;
    for (int w = tid; w < words; w += kNmsThreads) {
      unsigned long long mask = mask_ws[(int64_t)n * words + w];
      if (mask == 0) continue;
      int slot = atomicAdd(&s_count, __popcll(mask));
      for (; mask != 0; mask &= mask - 1, ++slot) {
        const unsigned b = (unsigned)w * 64 + (unsigned)(__ffsll(mask) - 1);
        (slot < lds_slots ? lds_keys : keys)[slot] = b;
      }
    }
  }
  __syncthreads();
  const int M = s_count;
  if (M == 0 || max_out == 0) return;
  const bool on_cu = M <= lds_slots;   // (lds_slots is a power of two: the padded list fits as well)
  if (mask_ws == nullptr) {
    if (!on_cu)
      for (int i = tid; i < lds_slots; i += kNmsThreads) keys[i] = lds_keys[i];
  } else {
    for (int i = tid; i < M; i += kNmsThreads) {
      const unsigned b = (unsigned)(i < lds_slots ? lds_keys : keys)[i];
      (on_cu ? lds_keys : keys)[i] = key_of(bestv[b], b);
    }
  }
  __syncthreads();
  const int P = (int)next_pow2(M);
  if (on_cu) {
    if (P <= kNmsThreads) nms_on_cu<TB, 1>(bx, cls, o, lds_keys, image_base + n, M, P, max_out, iou_thr);
    else nms_on_cu<TB, kNmsPerThread>(bx, cls, o, lds_keys, image_base + n, M, P, max_out, iou_thr);
    return;
  }

  // ---- the list does not fit: phases 2 and 3 in the workspace ----
  for (int i = M + tid; i < P; i += kNmsThreads) keys[i] = ~0ull;
  for (int i = tid; i < M; i += kNmsThreads) sup[i] = 0;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < P; i += kNmsThreads) {
        const int l = i ^ j;
        if (l > i) {
          const unsigned long long a = keys[i], b = keys[l];
          const bool up = (i & k) == 0;
          if ((a > b) == up) { keys[i] = b; keys[l] = a; }
        }
      }
      __syncthreads();
    }
  }
  int kept = 0;  // every thread counts the kept boxes itself: one barrier per kept box
  const bool flags8 = (reinterpret_cast<uintptr_t>(sup) & 7u) == 0;
  for (int i = 0; i < M; ++i) {
    // (uniform: the flags were written before the last barrier.)  Runs of
    // suppressed candidates are skipped eight flags per read: the walk is a chain
    // of dependent reads, one per step.
    if (flags8 && (i & 7) == 0) {
      while (i + 8 <= M && *reinterpret_cast<const unsigned long long*>(sup + i) == 0x0101010101010101ull) i += 8;
      if (i >= M) break;
    }
    if (sup[i]) continue;
    if (kept >= max_out) break;
    const int bi = (int)(keys[i] & 0xffffffffu);
    if (tid == 0) {
      o[kept * 3 + 0] = image_base + n;   // (the image's number in the caller's batch)
      o[kept * 3 + 1] = cls[bi];
      o[kept * 3 + 2] = bi;
    }
    const Box4 a = norm_box(bx + (int64_t)bi * 4);
    const float area_a = box_area(a);
    for (int j = i + 1 + tid; j < M; j += kNmsThreads) {
      if (!sup[j]) {
        const Box4 b = norm_box(bx + (int64_t)(keys[j] & 0xffffffffu) * 4);
        if (iou_of(b, box_area(b), a, area_a) >= iou_thr) sup[j] = 1;
      }
    }
    ++kept;
    __syncthreads();
  }
}

}  // namespace

size_t nms_workspace_bytes(int N, int B) {
  const int64_t bpad = next_pow2(B);
  // keys (8 B) + suppression flags (1 B) per padded slot, class and best score per box (4 B each),
  // a word of threshold decisions per 64 boxes
  size_t bytes = (size_t)N * bpad * 8 + (size_t)N * ((B + 63) / 64) * 8;
  bytes += (size_t)N * B * 4 * 2;
  bytes += (size_t)N * bpad;
  return (bytes + 255) & ~(size_t)255;
}

size_t nms_class_offset(int N, int B) { return ((size_t)N * next_pow2(B) + (size_t)N * ((B + 63) / 64)) * 8; }
size_t nms_best_offset(int N, int B) { return nms_class_offset(N, B) + (size_t)N * B * 4; }

template <typename TB>
static hipError_t launch_nms_kernel(const void* boxes, const float* best, int N, int B, int max_out, float iou_thr, float score_thr,
                                    const unsigned long long* masks, int32_t* out, unsigned long long* keys, const int32_t* cls,
                                    unsigned char* sup, int64_t bpad, int image_base, hipStream_t stream) {
  // candidate list on the compute unit - first the keys (two exchange buffers of 8 B per
  // slot), then boxes and flags in their place (16 + 1 B per slot): up to 8192 candidates
  const int lds_slots = (int)(bpad < 8192 ? bpad : 8192);
  const size_t lds_bytes = (size_t)lds_slots * 17;
  static LdsLimit limit;
  const hipError_t e = limit.raise(reinterpret_cast<const void*>(nms_kernel<TB>), 8192 * 17);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(nms_kernel<TB>, dim3(N), dim3(kNmsThreads), lds_bytes, stream, (const TB*)boxes, best, B, max_out,
                     iou_thr, score_thr, masks, out, keys, cls, sup, bpad, lds_slots, image_base);
  return hipGetLastError();
}

hipError_t launch_nms(const void* boxes, DType boxes_dt, const void* scores, DType scores_dt, int N, int C, int B,
                      int max_out, float iou_thr, float score_thr, int32_t* out, void* workspace,
                      hipStream_t stream, int image_base, bool best_ready) {
  if (!boxes || !scores || !out || !workspace || N <= 0 || C <= 0 || B <= 0 || max_out < 0)
    return hipErrorInvalidValue;
  if ((reinterpret_cast<uintptr_t>(workspace) & 7u) != 0) return hipErrorInvalidValue;
  const int64_t bpad = next_pow2(B);
  if (bpad > (1 << 24)) return hipErrorInvalidValue;
  unsigned long long* keys = reinterpret_cast<unsigned long long*>(workspace);
  unsigned long long* masks = keys + (int64_t)N * bpad;
  int32_t* cls = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + nms_class_offset(N, B));
  float* best = reinterpret_cast<float*>(static_cast<char*>(workspace) + nms_best_offset(N, B));
  unsigned char* sup = reinterpret_cast<unsigned char*>(best + (int64_t)N * B);
  if (N > 65535) return hipErrorInvalidValue;
  const dim3 grid1((unsigned)((B + 63) / 64), (unsigned)N);
  if (!best_ready) switch (scores_dt) {
    case DT_F32: hipLaunchKernelGGL(nms_best_class_kernel<float>, grid1, dim3(256), 0, stream, (const float*)scores, C, B, score_thr, best, cls, masks); break;
    case DT_F16: hipLaunchKernelGGL(nms_best_class_kernel<f16_t>, grid1, dim3(256), 0, stream, (const f16_t*)scores, C, B, score_thr, best, cls, masks); break;
    case DT_BF16: hipLaunchKernelGGL(nms_best_class_kernel<bf16_t>, grid1, dim3(256), 0, stream, (const bf16_t*)scores, C, B, score_thr, best, cls, masks); break;
    default: return hipErrorInvalidValue;
  }
  switch (boxes_dt) {
    case DT_F32: return launch_nms_kernel<float>(boxes, best, N, B, max_out, iou_thr, score_thr, best_ready ? nullptr : masks, out, keys, cls, sup, bpad, image_base, stream);
    case DT_F16: return launch_nms_kernel<f16_t>(boxes, best, N, B, max_out, iou_thr, score_thr, best_ready ? nullptr : masks, out, keys, cls, sup, bpad, image_base, stream);
    case DT_BF16: return launch_nms_kernel<bf16_t>(boxes, best, N, B, max_out, iou_thr, score_thr, best_ready ? nullptr : masks, out, keys, cls, sup, bpad, image_base, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ohip
