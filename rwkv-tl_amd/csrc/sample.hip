// Token sampling on the device: repetition penalty, greedy argmax,
// temperature, top-k, top-p and the random draw for each row of logits, in
// one launch (semantics of demo/sampling.py:13-70).
//
// One 1024-thread workgroup per row; thread t holds logits [64 t, 64 t + 64)
// (f16 or f32 in memory, f32 in registers; V <= 65536), so the row is read
// from HBM once.
//
// * Thresholds. top-k keeps x >= the k-th largest value (ties kept, as
//   torch.topk's cutoff with `>=`); top-p keeps x >= the largest value y whose
//   inclusive mass sum_{x_j >= y} p_j exceeds top_p (the token at which the
//   descending cumulative mass first passes top_p is the last one kept, as in
//   sampling.py:62-68). Both are "largest value y with weight(x >= y) > W"
//   and are found exactly, without sorting: one pass of 256 equal-width bins
//   over [min, max] (the bin index is a monotone function of x), then radix
//   passes of up to 8 bits over the order-preserving integer key of x inside
//   the chosen bin, until one value remains.
// * Mass. exp(x - max) is summed in 64-bit fixed point (scale 2^40), so every
//   sum is exact and the result does not depend on summation order.
// * Draw. One Philox4x32-10 block (Salmon et al., "Parallel random numbers:
//   as easy as 1, 2, 3", SC'11) per row: key = seed, counter = (offset, row,
//   0). Its first 64 bits r pick target = floor(Z r / 2^64) in [0, Z), and the
//   token is the first index (vocabulary order) whose inclusive prefix of kept
//   mass exceeds target: inverse-CDF sampling of the kept distribution.
#include "rwkv7_common.h"

namespace rwkv7 {
namespace {

typedef unsigned long long u64;

constexpr int kSmpThreads = 1024;
constexpr int kSmpWaves = kSmpThreads / kWave;
constexpr int kSmpE = 64;                      // logits per thread
constexpr int kSmpMaxV = kSmpThreads * kSmpE;  // 65536
constexpr float kFix = 1099511627776.0f;       // 2^40
constexpr float kInf = __builtin_inff();
constexpr int kCandCap = 4096;                 // LDS candidates of a threshold's bin

struct SampleArgs {
  const void *logits;
  int64_t ld;
  int V;
  float temp, top_p, pen;
  int top_k;
  uint32_t seed_lo, seed_hi, off_lo, off_hi;
  uint32_t *seen;
  int64_t seen_ld;
  int update_seen;
  int64_t *out;
  float *probs;
  int64_t probs_ld;
};

struct SampleLds {
  u64 hist[256];
  u64 wu[kSmpWaves];
  float wa[kSmpWaves], wb[kSmpWaves];
  int wi[kSmpWaves];
  u64 cross_above;
  int cross_bin;
  int ncand;
  float cand[kCandCap];
};

RWKV7_DEV uint32_t okey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
RWKV7_DEV float okey_inv(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k); }

RWKV7_DEV u64 shfl_xor64(u64 v, int m) {
  const int lo = __shfl_xor((int)(uint32_t)v, m), hi = __shfl_xor((int)(uint32_t)(v >> 32), m);
  return (u64)(uint32_t)lo | ((u64)(uint32_t)hi << 32);
}
RWKV7_DEV u64 shfl_up64(u64 v, int d) {
  const int lo = __shfl_up((int)(uint32_t)v, d), hi = __shfl_up((int)(uint32_t)(v >> 32), d);
  return (u64)(uint32_t)lo | ((u64)(uint32_t)hi << 32);
}
RWKV7_DEV u64 shfl_down64(u64 v, int d) {
  const int lo = __shfl_down((int)(uint32_t)v, d), hi = __shfl_down((int)(uint32_t)(v >> 32), d);
  return (u64)(uint32_t)lo | ((u64)(uint32_t)hi << 32);
}

// The compiler would otherwise keep per-element values (64 u64 weights, 64
// keys) live from one pass to the next instead of recomputing them from the 64
// logits, which overflows the 128 VGPRs of a 1024-thread workgroup: each pass
// reads its constants through this opaque copy.
RWKV7_DEV float opaque(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

RWKV7_DEV u64 mass(float x, float m) { return (u64)(__expf(x - m) * kFix); }

RWKV7_DEV bool better(float v, int i, float bv, int bi) { return v > bv || (v == bv && i < bi); }

// Block (max value, lowest index among ties); every thread gets the result.
RWKV7_DEV void block_argmax(float &v, int &i, SampleLds &s) {
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    const float ov = __shfl_xor(v, m);
    const int oi = __shfl_xor(i, m);
    if (better(ov, oi, v, i)) v = ov, i = oi;
  }
  const int w = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) s.wa[w] = v, s.wi[w] = i;
  __syncthreads();
  v = s.wa[0], i = s.wi[0];
  for (int j = 1; j < kSmpWaves; ++j)
    if (better(s.wa[j], s.wi[j], v, i)) v = s.wa[j], i = s.wi[j];
  __syncthreads();
}

RWKV7_DEV void block_minmax(float &lo, float &hi, SampleLds &s) {
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    lo = fminf(lo, __shfl_xor(lo, m));
    hi = fmaxf(hi, __shfl_xor(hi, m));
  }
  const int w = threadIdx.x / kWave;
  if (threadIdx.x % kWave == 0) s.wa[w] = lo, s.wb[w] = hi;
  __syncthreads();
  lo = s.wa[0], hi = s.wb[0];
  for (int j = 1; j < kSmpWaves; ++j) lo = fminf(lo, s.wa[j]), hi = fmaxf(hi, s.wb[j]);
  __syncthreads();
}

// Exclusive prefix of x over the block in thread order, and the block total.
RWKV7_DEV u64 block_excl_scan(u64 x, u64 &total, SampleLds &s) {
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  u64 inc = x;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const u64 o = shfl_up64(inc, d);
    if (lane >= d) inc += o;
  }
  if (lane == kWave - 1) s.wu[w] = inc;
  __syncthreads();
  u64 base = 0, tot = 0;
  for (int j = 0; j < kSmpWaves; ++j) {
    const u64 o = s.wu[j];
    base += j < w ? o : 0ull;
    tot += o;
  }
  __syncthreads();
  total = tot;
  return base + inc - x;
}

// Over s.hist, the largest bin b with above + sum_{b' >= b} hist[b'] > W.
// Sets s.cross_bin = b (-1 if none) and s.cross_above = above + sum_{b' > b}.
RWKV7_DEV void find_cross(SampleLds &s, u64 above, u64 W) {
  if (threadIdx.x < kWave) {
    const int L = threadIdx.x;
    const u64 h[4] = {s.hist[4 * L], s.hist[4 * L + 1], s.hist[4 * L + 2], s.hist[4 * L + 3]};
    const u64 own = (h[0] + h[1]) + (h[2] + h[3]);
    u64 suf = own;  // sum over bins >= 4 L
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const u64 o = shfl_down64(suf, d);
      if (L + d < kWave) suf += o;
    }
    // suf does not increase with L, so the lanes that pass form a prefix
    const u64 mask = __ballot(above + suf > W);
    if (mask == 0) {
      if (L == 0) s.cross_bin = -1;
    } else if (L == 63 - __clzll(mask)) {
      u64 acc = above + suf - own;  // <= W: the lane above failed
      int b = 4 * L;
      for (int j = 3; j >= 0; --j) {
        if (acc + h[j] > W) {
          b = 4 * L + j;
          break;
        }
        acc += h[j];
      }
      s.cross_bin = b;
      s.cross_above = acc;
    }
  }
  __syncthreads();
}

// Largest value y among the elements x >= lo (lo > -inf; hi their maximum) with
// sum over x >= y of wt(x) > W, where wt(x) = 1 (MASS false) or mass(x, m).
// If the total is <= W, lo. Each thread holds E elements (-inf: none).
//
// One pass of 256 equal-width bins over [lo, hi] picks the bin that holds y;
// its elements are copied to LDS (when there are at most kCandCap of them),
// and radix passes of up to 8 bits over their order-preserving keys narrow the
// key range to one value. A larger bin is narrowed the same way straight from
// the registers.
template <bool MASS, int E>
RWKV7_DEV float select_gt(const float (&l)[E], float lo, float hi, float m, u64 W, SampleLds &s) {
  auto wt = [](float x, float mm) -> u64 { return MASS ? mass(x, mm) : 1ull; };
  if (!(lo < hi)) return lo;
  // pass 0: equal-width bins over [lo, hi]
  const float scale = fminf(256.f / (hi - lo), 3.0e38f);  // finite, so (lo - lo) * scale == 0
  auto lbin = [](float x, float o, float sc) { return (int)fminf(255.f, (x - o) * sc); };
  for (int i = threadIdx.x; i < 256; i += kSmpThreads) s.hist[i] = 0;
  if (threadIdx.x == 0) s.ncand = 0;
  __syncthreads();
  {
    const float mo = opaque(m);
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (l[e] > -kInf && l[e] >= lo) atomicAdd(&s.hist[lbin(l[e], lo, scale)], wt(l[e], mo));
  }
  __syncthreads();
  find_cross(s, 0, W);
  const int b0 = s.cross_bin;
  if (b0 < 0) return lo;
  u64 above = s.cross_above;
  // the elements of bin b0: their range, and a copy in LDS
  float nlo = kInf, nhi = -kInf;
  {
    const float lo2 = opaque(lo), sc2 = opaque(scale);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (l[e] > -kInf && l[e] >= lo2 && lbin(l[e], lo2, sc2) == b0) {
        nlo = fminf(nlo, l[e]), nhi = fmaxf(nhi, l[e]);
        const int slot = atomicAdd(&s.ncand, 1);
        if (slot < kCandCap) s.cand[slot] = l[e];
      }
    }
  }
  block_minmax(nlo, nhi, s);  // its barriers order the copy and the cross_bin reads before what follows
  const int ncand = s.ncand;
  const bool from_lds = ncand <= kCandCap;  // block-uniform
  // radix passes over the keys in [kl, kh]: the elements of bin b0
  uint32_t kl = okey(nlo), kh = okey(nhi);
  while (kl != kh) {
    const int top = 31 - __clz(kl ^ kh);  // highest differing bit
    const int sh = max(0, top - 7);
    const uint32_t dmask = (1u << (top - sh + 1)) - 1u;
    for (int i = threadIdx.x; i < 256; i += kSmpThreads) s.hist[i] = 0;
    __syncthreads();
    const float zero = opaque(0.f), mo = opaque(m);
    if (from_lds) {
      for (int i = threadIdx.x; i < ncand; i += kSmpThreads) {
        const float x = s.cand[i];
        const uint32_t k = okey(x);
        if (k >= kl && k <= kh) atomicAdd(&s.hist[(k >> sh) & dmask], wt(x, mo));
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint32_t k = okey(l[e] + zero);  // + 0 keeps the value (no -0 is left)
        if (l[e] > -kInf && k >= kl && k <= kh) atomicAdd(&s.hist[(k >> sh) & dmask], wt(l[e], mo));
      }
    }
    __syncthreads();
    find_cross(s, above, W);
    const int b = s.cross_bin;
    above = s.cross_above;
    __syncthreads();
    if (b < 0) break;  // unreachable: above <= W < above + weight([kl, kh]) holds here
    const uint32_t keep_hi = top == 31 ? 0u : (0xffffffffu << (top + 1));
    const uint32_t nl = (kl & keep_hi) | ((uint32_t)b << sh);
    const uint32_t nh = nl | ((1u << sh) - 1u);
    kl = max(kl, nl);
    kh = min(kh, nh);
  }
  return okey_inv(kl);
}

RWKV7_DEV void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const u64 p0 = (u64)0xD2511F53u * c[0], p1 = (u64)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0, n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[0] = n0, c[1] = (uint32_t)p1, c[2] = n2, c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u, k1 += 0xBB67AE85u;
  }
}

// Logits 8..8c+7 of this thread's 64, as f32 (-inf past V). VEC: rows
// 16-byte aligned and V % 8 == 0, so each 8-logit chunk is whole 16-byte
// loads or wholly past V. FMT: 0 half, 1 f32, 2 bfloat16.
template <bool VEC, int FMT>
RWKV7_DEV void load8(const void *row_ptr, int i0, int V, float *f) {
  constexpr bool F32 = FMT == 1, BF = FMT == 2;
  if (VEC) {
    if (F32) {
      const float4 *p = reinterpret_cast<const float4 *>(static_cast<const float *>(row_ptr) + i0);
      const float4 u = i0 < V ? p[0] : make_float4(-kInf, -kInf, -kInf, -kInf);
      const float4 v = i0 < V ? p[1] : make_float4(-kInf, -kInf, -kInf, -kInf);
      f[0] = u.x, f[1] = u.y, f[2] = u.z, f[3] = u.w, f[4] = v.x, f[5] = v.y, f[6] = v.z, f[7] = v.w;
    } else {
      const uint32_t ninf2 = BF ? 0xff80ff80u : 0xfc00fc00u;  // two 16-bit -inf
      const uint4 u = i0 < V ? *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(row_ptr) + i0)
                             : make_uint4(ninf2, ninf2, ninf2, ninf2);
      F16T<BF>::to_f8(u, f);
    }
  } else if (i0 + 8 <= V) {
    // rows of any alignment: whole eights in one copy (unaligned 16-byte loads;
    // eight narrow ones per eight touch a line each)
    if (F32) {
      __builtin_memcpy(f, static_cast<const float *>(row_ptr) + i0, 32);
    } else {
      uint4 u;
      __builtin_memcpy(&u, static_cast<const uint16_t *>(row_ptr) + i0, 16);
      F16T<BF>::to_f8(u, f);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = i0 + j;
      f[j] = i >= V  ? -kInf
             : F32 ? static_cast<const float *>(row_ptr)[i]
                   : F16T<BF>::to_f(static_cast<const uint16_t *>(row_ptr)[i]);
    }
  }
}

// Temperature-scaled sampling of one row from the E values each thread holds
// (-inf: none), the threads' values in vocabulary order thread by thread;
// idx(e) is the vocabulary index of this thread's e-th value. Top-k, top-p,
// the kept mass and the draw as described at the top; pr (optional) receives
// the kept distribution at the indices held. Returns the token on the one
// thread that draws it, -1 on the others.
// The top-p threshold when at most kWave values are kept: the largest kept
// value y with sum_{x >= y} mass(x) > W is the value at the first position
// of the descending order whose running mass exceeds W (a tie group's
// members share the value, so where in the group that position falls does
// not matter). The kept values are compacted to LDS, and wave 0 sorts them
// (bitonic, one per lane), forms the running masses and picks that value.
// Returns false (and does nothing else) when more values are kept.
template <int E>
RWKV7_DEV bool top_p_in_wave(const float (&l)[E], float m, float top_p, float &thr, SampleLds &s) {
  int own = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) own += l[e] > -kInf;
  u64 total;
  int at = (int)block_excl_scan((u64)own, total, s);
  if (total > (u64)kWave) return false;  // block-uniform
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (l[e] > -kInf) s.cand[at++] = l[e];
  __syncthreads();
  if (threadIdx.x < kWave) {
    const int L = threadIdx.x;
    float v = L < (int)total ? s.cand[L] : -kInf;
    const float mo = opaque(m);
    u64 z = v > -kInf ? mass(v, mo) : 0ull;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) z += shfl_xor64(z, d);
    const u64 W = (u64)((double)top_p * (double)z);
#pragma unroll
    for (int k = 2; k <= kWave; k <<= 1) {  // descending bitonic sort over the lanes
#pragma unroll
      for (int j = k >> 1; j > 0; j >>= 1) {
        const float o = __shfl_xor(v, j);
        const bool take_max = ((L & j) == 0) == ((L & k) == 0);
        v = take_max ? fmaxf(v, o) : fminf(v, o);
      }
    }
    u64 c = v > -kInf ? mass(v, mo) : 0ull;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const u64 o = shfl_up64(c, d);
      if (L >= d) c += o;
    }
    const u64 pass = __ballot(c > W);  // nonzero: the last lane holds z > W
    const int first = __ffsll((unsigned long long)pass) - 1;
    const float y = __shfl(v, first);
    if (L == 0) s.wa[0] = y;
  }
  __syncthreads();
  thr = s.wa[0];
  __syncthreads();
  return true;
}

// FLOOR: before the top-k selection, bound the k-th largest value from below
// by the k-th largest of the threads' maxima (a saving when every thread holds
// many values, as in the one-workgroup kernel).
template <int E, bool FLOOR, class Idx>
RWKV7_DEV int draw_tempered(float (&l)[E], Idx idx, const SampleArgs &a, int row, float *pr, SampleLds &s) {
  const int V = a.V;
  float lo = kInf, m = -kInf, tmax = -kInf;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (l[e] > -kInf) lo = fminf(lo, l[e]), tmax = fmaxf(tmax, l[e]);
  m = tmax;
  block_minmax(lo, m, s);
  float thr = -kInf;  // tokens with x >= thr stay
  bool small = false;  // at most kWave tokens left after top-k
  if (a.top_k > 0 && a.top_k < V) {  // sampling.py:56-60
    // The k-th largest value is at least the k-th largest of the threads'
    // maxima when k threads hold values: only values from there up take part.
    float floor_k = lo;
    if (FLOOR && __syncthreads_count(tmax > -kInf) >= a.top_k) {
      float tl = tmax > -kInf ? tmax : kInf, th = tmax;
      block_minmax(tl, th, s);
      const float tv[1] = {tmax};
      floor_k = select_gt<false, 1>(tv, tl, th, m, (u64)(a.top_k - 1), s);
    }
    thr = select_gt<false, E>(l, floor_k, m, m, (u64)(a.top_k - 1), s);
    lo = thr;  // the smallest value top-k keeps
    small = a.top_k <= kWave;
  }
  if (a.top_p < 1.f) {  // sampling.py:62-68
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (l[e] < thr) l[e] = -kInf;
    float tp;
    if (small && top_p_in_wave<E>(l, m, a.top_p, tp, s)) {
      thr = tp;
    } else {
      u64 own = 0, z = 0;
      const float mo = opaque(m);
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (l[e] > -kInf) own += mass(l[e], mo);
      block_excl_scan(own, z, s);
      thr = select_gt<true, E>(l, lo, m, m, (u64)((double)a.top_p * (double)z), s);
    }
  }
  u64 own = 0, z = 0;
  {
    const float m1 = opaque(m);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (l[e] < thr) l[e] = -kInf;
      if (l[e] > -kInf) own += mass(l[e], m1);
    }
  }
  const u64 excl = block_excl_scan(own, z, s);
  uint32_t c[4] = {a.off_lo, a.off_hi, (uint32_t)row, 0u};
  philox4x32_10(c, a.seed_lo, a.seed_hi);
  const u64 target = __umul64hi(z, (u64)c[0] | ((u64)c[1] << 32));  // in [0, z)
  int token = -1;  // exactly one thread finds it: z >= 2^40, since the maximum is always kept
  if (excl <= target && target < excl + own) {
    u64 acc = excl;
    const float m2 = opaque(m);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (l[e] > -kInf) acc += mass(l[e], m2);
      if (token < 0 && acc > target) token = idx(e);
    }
  }
  if (pr) {
    const float inv = 1.f / (float)z, m3 = opaque(m);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = idx(e);
      if (i < V) pr[i] = l[e] > -kInf ? (float)mass(l[e], m3) * inv : 0.f;
    }
  }
  return token;
}

// The whole row on one workgroup (thread t holds logits 64 t .. 64 t + 63).
// Returns the token on the thread that holds it (every thread for greedy).
template <bool VEC, int FMT>
RWKV7_DEV int sample_row(const SampleArgs &a, int row, SampleLds &s) {
  const int base = threadIdx.x * kSmpE, V = a.V;
  const void *src = static_cast<const char *>(a.logits) + (int64_t)row * a.ld * (FMT == 1 ? 4 : 2);
  float l[kSmpE];
#pragma unroll
  for (int c = 0; c < kSmpE / 8; ++c) load8<VEC, FMT>(src, base + 8 * c, V, &l[8 * c]);
  // repetition penalty (sampling.py:44-47), applied once per seen token
  if (a.seen && a.pen != 1.f) {
    const uint32_t *sr = a.seen + (int64_t)row * a.seen_ld;
    const int nw = (V + 31) / 32;
    const uint32_t m0 = 2 * threadIdx.x < nw ? sr[2 * threadIdx.x] : 0u;
    const uint32_t m1 = 2 * threadIdx.x + 1 < nw ? sr[2 * threadIdx.x + 1] : 0u;
#pragma unroll
    for (int e = 0; e < kSmpE; ++e) {
      if (((e < 32 ? m0 : m1) >> (e & 31)) & 1u) l[e] = l[e] > 0.f ? l[e] / a.pen : l[e] * a.pen;
    }
  }
#pragma unroll
  for (int e = 0; e < kSmpE; ++e) l[e] = l[e] + 0.f;  // -0 -> +0: one key per value

  float *pr = a.probs ? a.probs + (int64_t)row * a.probs_ld : nullptr;
  if (!(a.temp > 0.f)) {
    // greedy: argmax, first index among ties (sampling.py:49-50)
    float v = -kInf;
    int vi = 0x7fffffff;
#pragma unroll
    for (int e = 0; e < kSmpE; ++e)
      if (better(l[e], base + e, v, vi)) v = l[e], vi = base + e;
    block_argmax(v, vi, s);
    const int token = vi < V ? vi : 0;  // only a row of NaNs leaves vi past V
    if (pr) {
#pragma unroll
      for (int e = 0; e < kSmpE; ++e)
        if (base + e < V) pr[base + e] = base + e == token ? 1.f : 0.f;
    }
    return threadIdx.x == 0 ? token : -1;
  }
#pragma unroll
  for (int e = 0; e < kSmpE; ++e) l[e] = l[e] / a.temp;
  return draw_tempered<kSmpE, true>(l, [base](int e) { return base + e; }, a, row, pr, s);
}

RWKV7_DEV void put_token(const SampleArgs &a, int row, int token) {
  if (token >= 0) {
    a.out[row] = token;
    if (a.update_seen) atomicOr(a.seen + (int64_t)row * a.seen_ld + token / 32, 1u << (token % 32));
  }
}

template <bool VEC, int FMT>
__global__ __launch_bounds__(kSmpThreads) void sample_kernel(SampleArgs a) {
  __shared__ SampleLds s;
  put_token(a, blockIdx.x, sample_row<VEC, FMT>(a, blockIdx.x, s));
}

// ---------------------------------------------------------------------------
// Top-k over many CUs (temperature > 0, 1 <= top_k <= kCandMax, no probs): the
// row is cut into equal slices of at most kCandSlice logits, one wave each
// (sample_cand_kernel; equal also over its lanes, in whole eights, so that no
// slice is left with too few maxima for a sharp floor), that keep a superset of the values top-k can keep, in
// index order; sample_finish_kernel finds the exact thresholds among them and
// draws. The candidates hold the same values at the same vocabulary positions
// as in the one-workgroup kernel and every sum is exact, so the token is the
// same.
//
// What bounds the two kernels is not the row's bytes (128 KB) but the chain of
// dependent selections. As histogram passes of a 1024-thread workgroup, with
// barriers between them, they took 15.1 + 23.8 us at 16 f16 rows of V = 65536,
// top-k 50, top-p 0.9; now 8.2 + 12.7 (whole calls, 16 f16 rows: V = 65536 top-k 1
// 30.2 -> 15.3, top-k 100 38.3 -> 22.5; V = 5000 top-k 50 25.0 -> 19.4, top-k 100
// 22.9 -> 18.8, top-k 128 69.6 -> 71.6 where a tie group sends rows to
// sample_row). A wave alone finds the k-th largest of the values its lanes hold
// with a ballot per bit (kth_key), no LDS and no barrier, so:
// * a slice's floor is the top_k-th largest of 128 maxima, two of each lane, its
//   odd and even fours of values (from top_k = 65 of the 512 maxima of 4): at
//   least top_k values of the slice reach it, so the row's top_k-th largest does
//   too, and 1.1-1.2 top_k values pass (more than kSliceCap, at top_k near it:
//   the slice's exact top_k-th largest instead);
// * the row's floor is the larger of two bounds on the row's top_k-th largest:
//   the largest slice floor, and the smallest over the slices of their
//   ceil(top_k / slices)-th largest of the 128 maxima (each slice has that many
//   values from there up) -- a few hundred of the candidates pass it;
// * if at most kFinMax pass, wave 0 holds them, eight per lane, and takes the
//   exact top-k threshold, the top-p threshold and the draw by itself; else the
//   workgroup runs draw_tempered on all candidates.
// A slice with more than kSliceCap values at its floor (a tie group) marks its
// count -1, and the row is sampled by sample_row instead.
// ---------------------------------------------------------------------------
constexpr int kCandE = 32;                   // logits per lane of a slice
constexpr int kCandSlice = kCandE * kWave;   // 2048
constexpr int kCandMax = 128;                // the largest top_k, and the coarse maxima of a slice
constexpr int kSliceCap = 128;               // candidates kept per slice
constexpr int kFloorLow = 12;                // lowest bit of a floor's key that is decided
constexpr int kSliceSel = 256;               // values at the floor among which a wave selects again
constexpr int kCandSlices = kSmpMaxV / kCandSlice;
constexpr int kFinE = kCandSlices * kSliceCap / kSmpThreads;  // candidates per thread in the finish
constexpr int kFinMax = 512;                 // candidates wave 0 finishes by itself
static_assert(kFinE == 4 && kCandSlices == 32, "a half wave per slice in the finish");

struct CandBuf {
  int *cnt;          // [B][G]: candidates of each slice, -1 when more than kSliceCap
  uint32_t *floors;  // [B][G][2]: keys of the slice's two bounds
  float *val;        // [B][G][kSliceCap]
  int *idx;          // [B][G][kSliceCap]
  int G;
};

// The key of a value in the order-preserving integer order, 0 for one that is
// not there (-inf or NaN).
RWKV7_DEV uint32_t vkey(float x) { return x > -kInf ? okey(x) : 0u; }

// The k-th largest (k >= 1) of the N keys each lane of the wave holds, 0 when
// fewer than k are nonzero: bit by bit, the largest key that k of them reach.
// With LOW > 0 down to that bit only: a key that k of them reach, less than
// 2^LOW below. Each bit is a chain of ballots and scalar counts. t and bit:
// where to start, the bits above `bit` that all nonzero keys share.
template <int N, int LOW = 0>
RWKV7_DEV uint32_t kth_key(const uint32_t (&key)[N], int k, uint32_t t = 0, int bit = 31) {
#pragma unroll 1
  for (; bit >= LOW; --bit) {
    const uint32_t c = t | (1u << bit);
    int n = 0;
#pragma unroll
    for (int e = 0; e < N; ++e) n += __popcll(__ballot(key[e] >= c));
    if (n >= k) t = c;
  }
  return t;
}

// VEC: 16-byte loads.
template <bool VEC, int FMT>
__global__ __launch_bounds__(256) void sample_cand_kernel(SampleArgs a, CandBuf cb) {
  __shared__ float s_sel[4][kSliceSel];
  const int lane = threadIdx.x & 63, g = 4 * blockIdx.x + (threadIdx.x >> 6), row = blockIdx.y, V = a.V;
  if (g >= cb.G) return;
  const void *src = static_cast<const char *>(a.logits) + (int64_t)row * a.ld * (FMT == 1 ? 4 : 2);
  // this lane's eights of logits, at most kCandE / 8 of them
  const int n8 = (V + 7) / 8, lanes = kWave * cb.G, b0 = (kWave * g + lane) * n8 / lanes,
            b1 = (kWave * g + lane + 1) * n8 / lanes, i0 = 8 * b0;
  float l[kCandE];
#pragma unroll
  for (int c = 0; c < kCandE / 8; ++c) load8<VEC, FMT>(src, b0 + c < b1 ? i0 + 8 * c : V, V, &l[8 * c]);
  if (a.seen && a.pen != 1.f) {  // the same operations, in the same order, as sample_row
    const uint32_t *sr = a.seen + (int64_t)row * a.seen_ld;
    const int nw = (V + 31) / 32, w0 = i0 >> 5;
    const uint64_t two = (uint64_t)(w0 < nw ? sr[w0] : 0u) | ((uint64_t)(w0 + 1 < nw ? sr[w0 + 1] : 0u) << 32);
    const uint32_t w = (uint32_t)(two >> (i0 & 31));
#pragma unroll
    for (int e = 0; e < kCandE; ++e)
      if ((w >> e) & 1u) l[e] = l[e] > 0.f ? l[e] / a.pen : l[e] * a.pen;
  }
#pragma unroll
  for (int e = 0; e < kCandE; ++e) l[e] = (l[e] + 0.f) / a.temp;
  // maxima of the lane's fours, then of its odd and even fours (its halves would
  // be empty for lanes with sixteen values)
  uint32_t pk[8], hk[2];
#pragma unroll
  for (int q = 0; q < 8; ++q) pk[q] = vkey(fmaxf(fmaxf(l[4 * q], l[4 * q + 1]), fmaxf(l[4 * q + 2], l[4 * q + 3])));
#pragma unroll
  for (int h = 0; h < 2; ++h) hk[h] = max(max(pk[h], pk[h + 2]), max(pk[h + 4], pk[h + 6]));
  // (floors to 2^-11 of a value; top_k 1: the largest; the second bound only
  // where the slices' candidates can pass what one wave finishes)
  uint32_t fl, few = 0u;
  if (a.top_k == 1) {
    fl = max(hk[0], hk[1]);
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) fl = max(fl, (uint32_t)__shfl_xor((int)fl, d));
  } else {
    fl = a.top_k <= kWave ? kth_key<2, kFloorLow>(hk, a.top_k) : kth_key<8, kFloorLow>(pk, a.top_k);
    if (cb.G * kSliceCap > kFinMax) few = kth_key<2, kFloorLow>(hk, (a.top_k + cb.G - 1) / cb.G);
  }
  float thr = fl ? okey_inv(fl) : -kInf;
  int own, inc, total;  // this lane's kept values, their inclusive prefix over the lanes, the slice's
  auto count = [&]() {
    own = 0;
#pragma unroll
    for (int e = 0; e < kCandE; ++e) own += l[e] > -kInf && l[e] >= thr;
    inc = own;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int o = __shfl_up(inc, d);
      if (lane >= d) inc += o;
    }
    total = __shfl(inc, kWave - 1);
  };
  count();
  if (total > kSliceCap) {  // the slice's exact top_k-th largest (top_k near kCandMax, or ties)
    uint32_t k;
    if (total <= kSliceSel) {
      // among the values at the floor, gathered over the lanes: an eighth of the
      // ballots that all values take (16 rows of 5000 f16 logits, top-k 127:
      // a call 38.1 -> 25.5 us)
      constexpr int N = kSliceSel / kWave;
      float *sel = s_sel[threadIdx.x >> 6];
      int at = inc - own;
#pragma unroll
      for (int e = 0; e < kCandE; ++e)
        if (l[e] > -kInf && l[e] >= thr) sel[at++] = l[e];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // one wave's own LDS
      uint32_t key[N];
#pragma unroll
      for (int e = 0; e < N; ++e) key[e] = lane + kWave * e < total ? vkey(sel[lane + kWave * e]) : 0u;
      k = kth_key<N>(key, a.top_k);
    } else {
      uint32_t key[kCandE];
#pragma unroll
      for (int e = 0; e < kCandE; ++e) key[e] = vkey(l[e]);
      k = kth_key<kCandE>(key, a.top_k);
    }
    thr = k ? okey_inv(k) : -kInf;
    count();
  }
  const int64_t slot = (int64_t)row * cb.G + g;
  if (lane == 0) {
    cb.cnt[slot] = total <= kSliceCap ? total : -1;
    cb.floors[2 * slot] = fl;
    cb.floors[2 * slot + 1] = few;
  }
  if (total > kSliceCap) return;
  int64_t at = slot * kSliceCap + inc - own;
#pragma unroll
  for (int e = 0; e < kCandE; ++e) {
    if (l[e] > -kInf && l[e] >= thr) {
      cb.val[at] = l[e];
      cb.idx[at] = i0 + e;
      ++at;
    }
  }
}

RWKV7_DEV u64 wave_sum64(u64 v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) v += shfl_xor64(v, d);
  return v;
}

// draw_tempered for the values wave 0 holds (kFinMax / 64 per lane, in
// vocabulary order lane by lane; -inf: none), by that wave alone. buf: kFinMax
// floats of LDS. Returns the token on the lane that draws it, -1 on the others.
template <int N>
RWKV7_DEV int draw_in_wave(float (&l)[N], const int (&ix)[N], const SampleArgs &a, int row, float *buf) {
  const int L = threadIdx.x;
  uint32_t key[N];
  float m = -kInf;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    key[e] = vkey(l[e]);
    m = fmaxf(m, l[e]);
  }
  uint32_t lo = ~0u;  // the smallest key there is: above the highest bit it and m's differ in, all agree
#pragma unroll
  for (int e = 0; e < N; ++e) lo = min(lo, key[e] ? key[e] : ~0u);
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    m = fmaxf(m, __shfl_xor(m, d));
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, d));
  }
  const uint32_t hi = vkey(m);
  uint32_t tk = hi;
  if (a.top_k > 1 && hi != lo) {
    const int bit = hi ? 31 - __clz((int)(hi ^ lo)) : 31;
    int have = 0;  // fewer than top_k: none is cut
#pragma unroll
    for (int e = 0; e < N; ++e) have += __popcll(__ballot(key[e] != 0u));
    tk = have < a.top_k ? 0u : kth_key<N>(key, a.top_k, bit == 31 ? 0u : hi & (~0u << (bit + 1)), bit);
  }
  float thr = tk ? okey_inv(tk) : -kInf;  // sampling.py:56-60
  int own = 0;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    if (!(l[e] >= thr)) l[e] = -kInf;
    own += l[e] > -kInf;
  }
  if (a.top_p < 1.f) {  // sampling.py:62-68
    int inc = own;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int o = __shfl_up(inc, d);
      if (L >= d) inc += o;
    }
    const int total = __shfl(inc, kWave - 1);
    u64 z = 0;
#pragma unroll
    for (int e = 0; e < N; ++e)
      if (l[e] > -kInf) z += mass(l[e], m);
    z = wave_sum64(z);
    const u64 W = (u64)((double)a.top_p * (double)z);
    if (total <= 2 * kWave) {  // sorted over the lanes (value i on lane i % 64), the first whose running mass exceeds W
      int at = inc - own;
#pragma unroll
      for (int e = 0; e < N; ++e)
        if (l[e] > -kInf) buf[at++] = l[e];
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      float v0 = L < total ? buf[L] : -kInf, v1 = L + kWave < total ? buf[L + kWave] : -kInf;
      const bool two = total > kWave;  // uniform
      auto cmp = [&](float &v, int i, int k, int j) {  // one descending bitonic step of value i against value i ^ j
        const float o = __shfl_xor(v, j);
        const bool take_max = ((i & j) == 0) == ((i & k) == 0);
        v = take_max ? fmaxf(v, o) : fminf(v, o);
      };
#pragma unroll
      for (int k = 2; k <= kWave; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
          cmp(v0, L, k, j);
          if (two) cmp(v1, L + kWave, k, j);
        }
      }
      if (two) {  // merge the two halves, sorted in opposite directions
        const float hi = fmaxf(v0, v1), lo = fminf(v0, v1);
        v0 = hi;
        v1 = lo;
#pragma unroll
        for (int j = kWave / 2; j > 0; j >>= 1) {
          cmp(v0, L, 2 * kWave, j);
          cmp(v1, L + kWave, 2 * kWave, j);
        }
      }
      auto scan = [&](float v) {
        u64 c = v > -kInf ? mass(v, m) : 0ull;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
          const u64 o = shfl_up64(c, d);
          if (L >= d) c += o;
        }
        return c;
      };
      const u64 c0 = scan(v0);
      u64 pass = __ballot(c0 > W);
      if (pass == 0 && two) {  // (one of them passes: the last value's running mass is z > W)
        const u64 c1 = scan(v1) + (u64)(uint32_t)__shfl((int)(uint32_t)c0, kWave - 1) +
                       ((u64)(uint32_t)__shfl((int)(uint32_t)(c0 >> 32), kWave - 1) << 32);
        pass = __ballot(c1 > W);
        v0 = v1;
      }
      thr = __shfl(v0, __ffsll((unsigned long long)pass) - 1);
    } else {  // the largest key whose mass from there up exceeds W, bit by bit
      uint32_t t = 0;
#pragma unroll 1
      for (int bit = 31; bit >= 0; --bit) {
        const uint32_t c = t | (1u << bit);
        u64 q = 0;
#pragma unroll
        for (int e = 0; e < N; ++e)
          if (l[e] > -kInf && key[e] >= c) q += mass(l[e], m);
        if (wave_sum64(q) > W) t = c;
      }
      thr = okey_inv(t);
    }
  }
  u64 own_z = 0;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    if (l[e] < thr) l[e] = -kInf;
    if (l[e] > -kInf) own_z += mass(l[e], m);
  }
  u64 inc = own_z;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const u64 o = shfl_up64(inc, d);
    if (L >= d) inc += o;
  }
  const u64 excl = inc - own_z, z = wave_sum64(own_z);
  uint32_t c[4] = {a.off_lo, a.off_hi, (uint32_t)row, 0u};
  philox4x32_10(c, a.seed_lo, a.seed_hi);
  const u64 target = __umul64hi(z, (u64)c[0] | ((u64)c[1] << 32));  // in [0, z)
  int token = -1;
  if (excl <= target && target < excl + own_z) {
    u64 acc = excl;
#pragma unroll
    for (int e = 0; e < N; ++e) {
      if (l[e] > -kInf) acc += mass(l[e], m);
      if (token < 0 && acc > target) token = ix[e];
    }
  }
  return token;
}

template <bool VEC, int FMT>
__global__ __launch_bounds__(kSmpThreads) void sample_finish_kernel(SampleArgs a, CandBuf cb) {
  __shared__ SampleLds s;
  __shared__ int s_wave[kSmpWaves + 1], s_ix[kFinMax];
  const int row = blockIdx.x, G = cb.G, t = threadIdx.x, lane = t & 63, wv = t >> 6;
  // half wave -> slice, four candidates per thread
  const int g = t >> 5, p0 = kFinE * (t & 31);
  const int64_t slot = (int64_t)row * G + min(g, G - 1);
  const int cnt = g < G ? cb.cnt[slot] : 0;
  if (__syncthreads_or(cnt < 0)) {  // a tie group overflowed a slice: the whole row here
    put_token(a, row, sample_row<VEC, FMT>(a, row, s));
    return;
  }
  float l[kFinE];
  int ix[kFinE];
  {
    // (all of a slice's places are readable; those past its count are dropped)
    const float4 v = p0 < cnt ? *reinterpret_cast<const float4 *>(cb.val + slot * kSliceCap + p0) : make_float4(0.f, 0.f, 0.f, 0.f);
    const int4 q = p0 < cnt ? *reinterpret_cast<const int4 *>(cb.idx + slot * kSliceCap + p0) : make_int4(0, 0, 0, 0);
    const float vv[4] = {v.x, v.y, v.z, v.w};
    const int qq[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < kFinE; ++e) {
      l[e] = p0 + e < cnt ? vv[e] : -kInf;
      ix[e] = p0 + e < cnt ? qq[e] : a.V;
    }
  }
  // the row's floor: every wave from the slices' bounds (lane -> slice)
  const int gl = min(lane & 31, G - 1);
  const uint32_t *fp = cb.floors + 2 * ((int64_t)row * G + gl);
  uint32_t top = fp[0], few = fp[1];
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) {
    top = max(top, (uint32_t)__shfl_xor((int)top, d));
    few = min(few, (uint32_t)__shfl_xor((int)few, d));
  }
  const uint32_t fkey = max(top, few);
  const float fl = fkey ? okey_inv(fkey) : -kInf;
  // candidates from the floor up, compacted in order
  int own = 0;
#pragma unroll
  for (int e = 0; e < kFinE; ++e) own += l[e] > -kInf && l[e] >= fl;
  int inc = own;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int o = __shfl_up(inc, d);
    if (lane >= d) inc += o;
  }
  if (lane == kWave - 1) s_wave[wv] = inc;
  __syncthreads();
  int base = 0, n = 0;
#pragma unroll
  for (int w = 0; w < kSmpWaves; ++w) {
    const int c = s_wave[w];
    base += w < wv ? c : 0;
    n += c;
  }
  if (n > kFinMax) {  // block-uniform
    put_token(a, row, draw_tempered<kFinE, false>(l, [&ix](int e) { return ix[e]; }, a, row, nullptr, s));
    return;
  }
  int at = base + inc - own;
#pragma unroll
  for (int e = 0; e < kFinE; ++e) {
    if (l[e] > -kInf && l[e] >= fl) {
      s.cand[at] = l[e];
      s_ix[at] = ix[e];
      ++at;
    }
  }
  __syncthreads();
  if (wv > 0) return;
  constexpr int N = kFinMax / kWave;
  float x[N];
  int xi[N];
#pragma unroll
  for (int e = 0; e < N; ++e) {
    const int d = N * lane + e;
    x[e] = d < n ? s.cand[d] : -kInf;
    xi[e] = d < n ? s_ix[d] : a.V;
  }
  put_token(a, row, draw_in_wave<N>(x, xi, a, row, s.cand + kFinMax));
}

}  // namespace
}  // namespace rwkv7

static int64_t cand_bytes(int B, int G) {
  auto al = [](int64_t x) { return (x + 255) / 256 * 256; };
  return al((int64_t)B * G * 4) + al((int64_t)B * G * 8) + 2 * al((int64_t)B * G * rwkv7::kSliceCap * 4);
}

extern "C" int64_t rwkv7_sample_workspace_bytes(int32_t B, int32_t V) {
  using namespace rwkv7;
  if (B < 1 || V < 1 || V > kSmpMaxV) return 0;
  return cand_bytes(B, (V + kCandSlice - 1) / kCandSlice);
}

extern "C" int rwkv7_sample(const void *logits, int32_t logits_dtype, int64_t ld, int32_t B, int32_t V, const rwkv7_sampling *p,
                            uint32_t *seen, int64_t seen_ld, int32_t update_seen, int64_t *out, float *probs,
                            int64_t probs_ld, void *workspace, int64_t workspace_bytes, void *stream) {
  using namespace rwkv7;
  if (!logits || !p || !out || B < 1 || (update_seen && !seen)) return RWKV7_EINVAL;
  if (logits_dtype < 0 || logits_dtype > 2) return RWKV7_EINVAL;
  if (V < 1 || V > kSmpMaxV || ld < V || (seen && seen_ld < (V + 31) / 32) || (probs && probs_ld < V))
    return RWKV7_ESHAPE;
  SampleArgs a;
  a.logits = logits;
  a.ld = ld;
  a.V = V;
  a.temp = p->temperature;
  a.top_p = p->top_p;
  a.pen = p->repetition_penalty;
  a.top_k = p->top_k;
  a.seed_lo = (uint32_t)p->seed, a.seed_hi = (uint32_t)(p->seed >> 32);
  a.off_lo = (uint32_t)p->offset, a.off_hi = (uint32_t)(p->offset >> 32);
  a.seen = seen;
  a.seen_ld = seen_ld;
  a.update_seen = update_seen;
  a.out = out;
  a.probs = probs;
  a.probs_ld = probs_ld;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const bool vec = reinterpret_cast<uintptr_t>(logits) % 16 == 0 && ld % 8 == 0 && V % 8 == 0;
  const int G = (V + kCandSlice - 1) / kCandSlice;
  const bool cand = workspace && workspace_bytes >= cand_bytes(B, G) && a.temp > 0.f && a.top_k >= 1 &&
                    a.top_k <= kCandMax && a.top_k < V && !probs && G >= 2;
  if (cand) {
    auto al = [](int64_t x) { return (x + 255) / 256 * 256; };
    char *w = static_cast<char *>(workspace);
    const int64_t c0 = al((int64_t)B * G * 4), c1 = c0 + al((int64_t)B * G * 8), nv = al((int64_t)B * G * kSliceCap * 4);
    CandBuf cb;
    cb.cnt = reinterpret_cast<int *>(w);
    cb.floors = reinterpret_cast<uint32_t *>(w + c0);
    cb.val = reinterpret_cast<float *>(w + c1);
    cb.idx = reinterpret_cast<int *>(w + c1 + nv);
    cb.G = G;
    const dim3 grid((G + 3) / 4, B);
    switch (logits_dtype) {
      case 0: vec ? sample_cand_kernel<true, 0><<<grid, 256, 0, st>>>(a, cb) : sample_cand_kernel<false, 0><<<grid, 256, 0, st>>>(a, cb); break;
      case 1: vec ? sample_cand_kernel<true, 1><<<grid, 256, 0, st>>>(a, cb) : sample_cand_kernel<false, 1><<<grid, 256, 0, st>>>(a, cb); break;
      default: vec ? sample_cand_kernel<true, 2><<<grid, 256, 0, st>>>(a, cb) : sample_cand_kernel<false, 2><<<grid, 256, 0, st>>>(a, cb); break;
    }
    RWKV7_CHECK_LAUNCH();
    switch (logits_dtype) {
      case 0: vec ? sample_finish_kernel<true, 0><<<B, kSmpThreads, 0, st>>>(a, cb) : sample_finish_kernel<false, 0><<<B, kSmpThreads, 0, st>>>(a, cb); break;
      case 1: vec ? sample_finish_kernel<true, 1><<<B, kSmpThreads, 0, st>>>(a, cb) : sample_finish_kernel<false, 1><<<B, kSmpThreads, 0, st>>>(a, cb); break;
      default: vec ? sample_finish_kernel<true, 2><<<B, kSmpThreads, 0, st>>>(a, cb) : sample_finish_kernel<false, 2><<<B, kSmpThreads, 0, st>>>(a, cb); break;
    }
    RWKV7_CHECK_LAUNCH();
    return RWKV7_OK;
  }
  switch (logits_dtype) {
    case 0: vec ? sample_kernel<true, 0><<<B, kSmpThreads, 0, st>>>(a) : sample_kernel<false, 0><<<B, kSmpThreads, 0, st>>>(a); break;
    case 1: vec ? sample_kernel<true, 1><<<B, kSmpThreads, 0, st>>>(a) : sample_kernel<false, 1><<<B, kSmpThreads, 0, st>>>(a); break;
    default: vec ? sample_kernel<true, 2><<<B, kSmpThreads, 0, st>>>(a) : sample_kernel<false, 2><<<B, kSmpThreads, 0, st>>>(a); break;
  }
  RWKV7_CHECK_LAUNCH();
  return RWKV7_OK;
}
