// MFMA GEMM on fragment-ordered operands: Y = epi(A W^T) for steps of 9 rows
// up to the large-M path with f32-grade activations.
//
// Both operands are stored as MFMA reads them, in 16-row x 32-k blocks of one
// contiguous KiB per 64-lane load: W in the model's fragment arena, A in split
// order (split_put8) by the kernels that produce it: the activations' 16-bit
// parts and their 16-bit remainders (split_hi_lo's two values). So a wave loads
// both operands straight into MFMA registers, and the main loop is loads and
// MFMAs: no LDS, no conversion, no barrier until the waves' partial tiles meet.
//
// At these sizes (M up to ~2000) a product is neither MFMA- nor HBM-bound but
// bound by the operand bytes that each CU pulls through its L1 (64 bytes per
// cycle) and by the round trips in a workgroup's life. The tiled kernels of
// gemm.hip (16 or 32 rows x 64 columns, A split and staged through LDS) moved
// more bytes per product and waited for load, LDS and product phases in turn.
// Here 8 waves share a tile as SM x SN sub-tiles of MB x NB blocks and SK
// slices of K: few rows take a small tile with K split over the eight waves
// (every load of the tile in flight at once), many rows a larger tile that
// reuses each byte more. The K slices' partials are summed in LDS in slice
// order, where the accumulator layout also becomes rows for vector stores.
#include "rwkv7_kernels.h"

#include <algorithm>

namespace rwkv7 {

constexpr int kFragProbs = 8;
constexpr int kFragThreads = 512;

struct FragGroup {
  GemmProb p[kFragProbs];
  int unit_begin[kFragProbs];  // first unit (column tile and K slice) of each problem
  int nprob, M, m_tiles;
  int items, per_xcd;  // tiles of all units, and of each XCD's run of them
  // K cut into `splits` (a power of two), each slice's f32 partial product
  // stored at Y + slice * part_stride floats: the next stage sums them
  int splits;
  int64_t part_stride;
};

// A workgroup's tile. The tiles of the group, row tiles of a unit together, are
// cut into eight equal runs, one per XCD (workgroups are dealt to the XCDs in
// turn): every XCD gets as many, and the row tiles of a unit read W from its
// L2. (Padded to eight units per problem instead, the 22 units of an r, k, v and
// LoRA group of 768 columns left two XCDs idle, and its LoRA tiles all ran on
// one: 656 rows 32.0 -> 13.2 us; of 1024 columns, 509 rows 27.3 -> 15.7.)
struct FragItem {
  int prob, unit, mt;  // unit -1: none
};
RWKV7_DEV FragItem frag_item(const FragGroup &g) {
  const int item = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= g.per_xcd || item >= g.items) return {0, -1, 0};
  const int u = item / g.m_tiles;
  int pi = 0;
#pragma unroll
  for (int i = 1; i < kFragProbs; ++i) pi += (i < g.nprob && u >= g.unit_begin[i]);
  return {pi, u - g.unit_begin[pi], item - u * g.m_tiles};
}

// The epilogue's value for one element (the add epilogue reads Y elsewhere).
RWKV7_DEV float frag_epi(int epi, float v) {
  switch (epi) {
    case GEPI_RELUSQ_F32:
    case GEPI_RELUSQ_SPLIT: {
      const float q = fmaxf(v, 0.f);
      return q * q;
    }
    case GEPI_TANH_F32:
    case GEPI_TANH_SPLIT: return tanhf(v);
    case GEPI_SIGM_F32:
    case GEPI_SIGM_SPLIT: return sigmoidf_(v);
    default: return v;
  }
}

// Output piece u of a thread: four columns of a row of the tile.
template <int BM, int BN>
RWKV7_DEV bool frag_piece(int u, int &row, int &col) {
  const int e = (int)threadIdx.x + kFragThreads * u;
  row = e / (BN / 4);
  col = 4 * (e % (BN / 4));
  return e < BM * BN / 4;
}
template <int BM, int BN>
constexpr int kFragPieces = BM * BN / 4 / kFragThreads > 0 ? BM * BN / 4 / kFragThreads : 1;

// The values an add epilogue accumulates into.
template <int BM, int BN>
RWKV7_DEV void frag_yres(const GemmProb &P, int M, int m0, int n0, float4 (&yres)[kFragPieces<BM, BN>]) {
#pragma unroll
  for (int u = 0; u < kFragPieces<BM, BN>; ++u) {
    int row, col;
    frag_piece<BM, BN>(u, row, col);
    yres[u] = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(P.Y) +
                                                (int64_t)min(m0 + row, M - 1) * P.ldy + min(n0 + col, P.N - 4));
  }
}

// A tile's SK partial products in LDS: summed in order, epilogue, stored.
template <int BM, int BN, int SK, bool BF>
RWKV7_DEV void frag_store(const FragGroup &g, const GemmProb &P, const float (*s_red)[BM][BN + 4],
                          const float4 (&yres)[kFragPieces<BM, BN>], int m0, int n0, int split) {
  constexpr int PPT = kFragPieces<BM, BN>;
  const int M = g.M, N = P.N, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const bool add = P.epi == GEPI_ADD_F32;
  const int epi = P.epi;
  if (epi >= GEPI_SPLIT) {
    // the next product's A: a wave per 16 x 32 block of the tile, one
    // contiguous KiB per part; columns up to the next k-step are zeros
    constexpr int NBLK = BM / 16 * (BN / 32);
#pragma unroll
    for (int q = 0; q < (NBLK + 7) / 8; ++q) {
      const int blk = wv + 8 * q, row = 16 * (blk / (BN / 32)) + (lane & 15), col = 32 * (blk % (BN / 32)) + 8 * (lane >> 4);
      const int m = m0 + row, n = n0 + col;
      if (blk >= NBLK || m >= M || n >= (N + 31) / 32 * 32) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
      for (int s = 0; s < SK; ++s) {
        const float4 x = *reinterpret_cast<const float4 *>(&s_red[s][row][col]);
        const float4 y = *reinterpret_cast<const float4 *>(&s_red[s][row][col + 4]);
        v[0] += x.x;
        v[1] += x.y;
        v[2] += x.z;
        v[3] += x.w;
        v[4] += y.x;
        v[5] += y.y;
        v[6] += y.z;
        v[7] += y.w;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = n + e < N ? frag_epi(epi, v[e]) : 0.f;
      split_put8<BF>(static_cast<uint16_t *>(P.Y), (N + 31) / 32, m, n, v);
    }
    return;
  }
  const bool vec = N % 4 == 0 && P.ldy % 4 == 0;
#pragma unroll
  for (int u = 0; u < PPT; ++u) {
    int row, col;
    if (!frag_piece<BM, BN>(u, row, col)) continue;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SK; ++s) {
      const float4 q = *reinterpret_cast<const float4 *>(&s_red[s][row][col]);
      v[0] += q.x;
      v[1] += q.y;
      v[2] += q.z;
      v[3] += q.w;
    }
    const int m = m0 + row, n = n0 + col;
    if (m >= M) continue;
    if (n >= N) continue;
    const int64_t o = (int64_t)m * P.ldy + n;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = frag_epi(epi, v[e]);
    if (epi == GEPI_F16) {
      uint16_t *y = static_cast<uint16_t *>(P.Y) + o;
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = F16T<BF>::from_f(v[e]);
      if (vec) {
        *reinterpret_cast<uint2 *>(y) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) y[e] = h[e];
      }
    } else {
      float *y = static_cast<float *>(P.Y) + split * g.part_stride + o;
      if (add) {
        v[0] += yres[u].x;
        v[1] += yres[u].y;
        v[2] += yres[u].z;
        v[3] += yres[u].w;
      }
      if (vec) {
        *reinterpret_cast<float4 *>(y) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) y[e] = v[e];
      }
    }
  }
}

template <int MB, int NB, int SM, int SN, int SK, int KB, bool BF>
__global__ __launch_bounds__(kFragThreads) void gemm_frag_kernel(FragGroup g) {
  constexpr int BM = 16 * MB * SM, BN = 16 * NB * SN, LD = BN + 4;
  static_assert(SM * SN * SK * 64 == kFragThreads, "eight waves");
  __shared__ __align__(16) float s_red[SK][BM][LD];

  const FragItem it = frag_item(g);
  if (it.unit < 0) return;
  const GemmProb &P = g.p[it.prob];
  const int N = P.N, M = g.M, S = g.splits, mt = it.mt;
  const int nt = it.unit / S, split = it.unit & (S - 1);
  const int m0 = mt * BM, n0 = nt * BN;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv % SM, wn = wv / SM % SN, wk = wv / (SM * SN);

  // operand blocks (rows and columns past the matrices are clamped to their
  // last block: products nobody stores)
  const int nks = (P.K + 31) / 32, per = (nks + SK * S - 1) / (SK * S);
  const int k0 = (split * SK + wk) * per, len = max(0, min(nks, k0 + per) - k0);
  // each wave and row tile starts elsewhere in its slice, so that the tiles of
  // a column do not ask for the same lines at once (128 rows of 3360 x 1024
  // 8.6 -> 7.7 us, 4096 x 1024 9.7 -> 8.6 us)
  const int rot = len > 0 ? (3 * mt + wv) % len : 0;
  const uint16_t *pa[MB], *pw[NB];
  const int mblk = (M + 15) / 16, nstrip = (N + 15) / 16;
#pragma unroll
  for (int i = 0; i < MB; ++i)
    pa[i] = P.A + (int64_t)min(m0 / 16 + wm * MB + i, mblk - 1) * nks * 1024 + lane * 8;
#pragma unroll
  for (int j = 0; j < NB; ++j) pw[j] = P.Wf + (int64_t)min(n0 / 16 + wn * NB + j, nstrip - 1) * P.nksf * 512 + lane * 8;

  uint4 a[2][KB][MB][2], w[2][KB][NB];
  auto load = [&](int k, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      int kk = min(k + b, len - 1) + rot;  // clamped: never multiplied past the slice
      kk = kk >= len ? kk - len : kk;
      kk = min(max(kk + k0, 0), nks - 1);  // (an empty slice loads something valid)
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        a[buf][b][i][0] = *reinterpret_cast<const uint4 *>(pa[i] + (int64_t)kk * 1024);
        a[buf][b][i][1] = *reinterpret_cast<const uint4 *>(pa[i] + (int64_t)kk * 1024 + 512);
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) w[buf][b][j] = *reinterpret_cast<const uint4 *>(pw[j] + (int64_t)kk * 512);
    }
  };
  floatx4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int k, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      if (k + b < len) {
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = mfma16<BF>(a[buf][b][i][pl], w[buf][b][j], acc[i][j]);
      }
    }
  };
  load(0, 0);
  load(KB, 1);
  // the values an add epilogue accumulates into, behind the first operands
  float4 yres[kFragPieces<BM, BN>];
  if (P.epi == GEPI_ADD_F32) frag_yres<BM, BN>(P, M, m0, n0, yres);
  __builtin_amdgcn_sched_barrier(0);
  for (int k = 0; k < len; k += 2 * KB) {
    compute(k, 0);
    load(k + 2 * KB, 0);
    __builtin_amdgcn_sched_barrier(0);
    compute(k + KB, 1);
    load(k + 3 * KB, 1);
    __builtin_amdgcn_sched_barrier(0);
  }

  // lane holds rows 4 (lane >> 4) + r of column lane & 15 of each block
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s_red[wk][16 * (wm * MB + i) + 4 * (lane >> 4) + r][16 * (wn * NB + j) + (lane & 15)] = acc[i][j][r];
  __syncthreads();
  frag_store<BM, BN, SK, BF>(g, P, s_red, yres, m0, n0, split);
}

// Many rows: the operands by LDS DMA. The register loads above pass every
// block through the CU's L1 once per wave that multiplies it -- twice for a
// 2 x 2 arrangement of sub-tiles, 32 KiB per k-step of a 64 x 128 tile, 512
// cycles of the L1's 64 bytes against 256 of MFMA. Here each block of a stage
// (SK k-steps, one per slice) is one DMA into a ring of NBUF stages, NBUF - 1
// ahead of the products, and the waves read it from LDS: a stage's fragments
// are read into one of two register sets while the previous stage's are
// multiplied.
template <int MB, int NB, int SM, int SN, int SK, int NBUF, bool BF>
__global__ __launch_bounds__(kFragThreads) void gemm_frag_ring_kernel(FragGroup g) {
  constexpr int BM = 16 * MB * SM, BN = 16 * NB * SN, LD = BN + 4;
  constexpr int NA = 2 * MB * SM, NW = NB * SN, BLK = SK * (NA + NW);  // blocks of a k-step, of a stage
  constexpr int WPS = 8 / SK, PA = NA / WPS, PW = NW / WPS;            // waves per k-step, blocks each loads
  static_assert(SM * SN * SK == 8 && NA % WPS == 0 && NW % WPS == 0, "eight waves, whole blocks each");
  constexpr int kVm = (NBUF - 2) * (PA + PW);  // this wave's DMAs behind the stage waited for
  static_assert(kVm < 64, "vmcnt field");
  constexpr int kWaitImm = 0x0F70 | (kVm & 15) | ((kVm >> 4) << 14);
  constexpr int kBytes = NBUF * BLK * 1024 > SK * BM * LD * 4 ? NBUF * BLK * 1024 : SK * BM * LD * 4;
  __shared__ __align__(1024) unsigned char smem[kBytes];

  const FragItem it = frag_item(g);
  if (it.unit < 0) return;
  const GemmProb &P = g.p[it.prob];
  const int N = P.N, M = g.M, S = g.splits, mt = it.mt;
  const int nt = it.unit / S, split = it.unit & (S - 1);
  const int m0 = mt * BM, n0 = nt * BN;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv % SM, wn = wv / SM % SN, wk = wv / (SM * SN);

  const int nks = (P.K + 31) / 32, per = (nks + S - 1) / S;
  const int k0 = split * per, len = max(0, min(nks, k0 + per) - k0);
  const int nst = (len + SK - 1) / SK;
  const int rot = nst > 0 ? 3 * mt % nst : 0;  // each row tile starts elsewhere, as above
  const int mblk = (M + 15) / 16, nstrip = (N + 15) / 16;
  // this wave's DMAs: blocks wq * PA .. of A (strip, part) and wq * PW .. of W,
  // k-step ws of the stage; rows past the matrices clamp to their last block
  const int ws = wv / WPS, wq = wv % WPS;
  const i32x4 ra = buffer_words(P.A, mblk * nks * 2048), rw = buffer_words(P.Wf, nstrip * P.nksf * 1024);
  int oa[PA], ow[PW];
#pragma unroll
  for (int u = 0; u < PA; ++u) {
    const int b = wq * PA + u;
    oa[u] = min(m0 / 16 + (b >> 1), mblk - 1) * nks * 2048 + (b & 1) * 1024 + lane * 16;
  }
#pragma unroll
  for (int u = 0; u < PW; ++u) ow[u] = min(n0 / 16 + wq * PW + u, nstrip - 1) * P.nksf * 1024 + lane * 16;
  auto stage_k = [&](int st) __attribute__((always_inline)) {  // first k-step of stage st, in the rotated order
    int t = min(st, nst - 1) + rot;
    t = t >= nst ? t - nst : t;
    return max(t, 0) * SK;
  };
  // (past the last stage the last one again, into a buffer nobody reads: the
  // vmcnt bookkeeping stays uniform)
  const uint32_t lds0 = lds_addr(smem) + (uint32_t)(ws * (NA + NW)) * 1024;
  auto issue = [&](int st, int buf) __attribute__((always_inline)) {
    const int kk = min(k0 + stage_k(st) + ws, nks - 1);
    const uint32_t base = lds0 + (uint32_t)buf * (BLK * 1024);
#pragma unroll
    for (int u = 0; u < PA; ++u) dma16(ra, base + (uint32_t)(wq * PA + u) * 1024, oa[u], kk * 2048);
#pragma unroll
    for (int u = 0; u < PW; ++u) dma16(rw, base + (uint32_t)(NA + wq * PW + u) * 1024, ow[u], kk * 1024);
  };
  floatx4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  struct Frags {
    uint4 a[MB][2], w[NB];
  };
  const unsigned char *fa = smem + (wk * (NA + NW) + wm * MB * 2) * 1024 + lane * 16;
  const unsigned char *fw = smem + (wk * (NA + NW) + NA + wn * NB) * 1024 + lane * 16;
  auto read = [&](Frags &f, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NB; ++j) f.w[j] = *reinterpret_cast<const uint4 *>(fw + buf * (BLK * 1024) + j * 1024);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int pl = 0; pl < 2; ++pl)
        f.a[i][pl] = *reinterpret_cast<const uint4 *>(fa + buf * (BLK * 1024) + (2 * i + pl) * 1024);
  };
  auto compute = [&](const Frags &f, int st) __attribute__((always_inline)) {
    if (stage_k(st) + wk >= len) return;  // the last stage may be short
#pragma unroll
    for (int pl = 0; pl < 2; ++pl)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma16<BF>(f.a[i][pl], f.w[j], acc[i][j]);
  };
  float4 yres[kFragPieces<BM, BN>];
  if (P.epi == GEPI_ADD_F32) frag_yres<BM, BN>(P, M, m0, n0, yres);
#pragma unroll
  for (int b = 0; b < NBUF - 1; ++b) issue(b, b);
  int buf = 0;
  // stage st has landed for every wave, and every read of the buffer that the
  // next DMA overwrites is complete
  auto arrive = [&](int st) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(kWaitImm);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue(st + NBUF - 1, buf == 0 ? NBUF - 1 : buf - 1);
  };
  auto next = [&]() __attribute__((always_inline)) { buf = buf == NBUF - 1 ? 0 : buf + 1; };
  Frags f0, f1;
  if (nst > 0) {
    arrive(0);
    read(f0, buf);
    next();
    int st = 1;
    for (; st + 1 < nst; st += 2) {
      arrive(st);
      read(f1, buf);
      next();
      __builtin_amdgcn_sched_barrier(0);
      compute(f0, st - 1);
      arrive(st + 1);
      read(f0, buf);
      next();
      __builtin_amdgcn_sched_barrier(0);
      compute(f1, st);
    }
    if (st < nst) {
      arrive(st);
      read(f1, buf);
      __builtin_amdgcn_sched_barrier(0);
      compute(f0, st - 1);
      compute(f1, st);
    } else {
      compute(f0, st - 1);
    }
  }
  // every DMA and every read of the ring is done before the partials replace it
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  float(*s_red)[BM][LD] = reinterpret_cast<float(*)[BM][LD]>(smem);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        s_red[wk][16 * (wm * MB + i) + 4 * (lane >> 4) + r][16 * (wn * NB + j) + (lane & 15)] = acc[i][j][r];
  __syncthreads();
  frag_store<BM, BN, SK, BF>(g, P, s_red, yres, m0, n0, split);
}

// Tiles, smallest first.
struct FragTile {
  int bm, bn;
};
constexpr FragTile kFragTiles[] = {{16, 32}, {32, 32}, {32, 64}, {64, 64}, {32, 128}, {64, 128}, {128, 128}};
constexpr int kFragOneRound = 6;  // the tiles before it; the last is for several rounds

static int64_t frag_units(const FragTile &t, int M, int N) {
  return (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
}

// The smallest tile whose workgroups all run at once (one per CU): a larger
// one leaves CUs idle, a smaller one moves more bytes per CU and runs in
// rounds (measured, us, 0.4B FFN key 4096 x 1024: 64 rows 32 x 32 7.9, 16 x 32
// 8.9, 32 x 64 8.7; 128 rows 32 x 64 9.1, 32 x 32 11.9, 64 x 64 11.4; 512 rows
// 64 x 128 16.1, 64 x 64 18.4; FFN value's and the 1.5B sizes order alike).
// Where none fits at once (an eighth more than the CUs still passes: two of the
// smaller tiles fit on one) the largest, with as few rows as M has.
//
// From 64 x 128 the operands come through LDS (gemm_frag_ring_kernel) if K is
// long enough to pay for filling the ring, and of several rounds each takes
// 128 x 128 if K covers its unoverlapped ends as well: two register-fed
// workgroups share a CU and hide theirs in each other. Measured, whole
// prefills in us, register-fed / ring: 1.5B 1 x 129 3371 / 2879, 4 x 64 3686 /
// 3331, 8 x 96 8989 / 8443, 0.4B 3 x 129 2404 / 2325, 1 x 509 2859 / 2827, 16 x
// 100 6484 / 6401; 0.1B (K 768) 8 x 60 1078 / 1052, but 16 x 96, three rounds,
// 2505 / 2683.
constexpr int kFragRingMinK = 512, kFragRoundsMinK = 1024;
static bool frag_ring(const GemmProb *probs, int nprob, int M, int min_k) {
  int k = 0;
  for (int q = 0; q < nprob; ++q) {
    const int64_t nks = (probs[q].K + 31) / 32, blocks = std::max((M + 15) / 16 * 2, (probs[q].N + 15) / 16);
    if (blocks * nks * 1024 > INT32_MAX) return false;  // the DMA's offsets are 32-bit
    k = std::max(k, probs[q].K);
  }
  return k >= min_k;
}
static int frag_tile(const GemmProb *probs, int nprob, int M, int cus) {
  for (int i = 0; i < kFragOneRound; ++i) {
    if (i == 4 && M > 32) continue;
    int64_t n = 0;
    for (int q = 0; q < nprob; ++q) n += frag_units(kFragTiles[i], M, probs[q].N);
    if (n <= cus + (i < 4 ? cus / 8 : 0)) return i;
  }
  return M <= 32 ? 4 : frag_ring(probs, nprob, M, kFragRoundsMinK) ? 6 : 5;
}

// K slices of a product whose partials the next stage can sum. Few rows and a
// long K leave each CU a small tile with all of K: its operands' bytes are the
// time. Cutting K lets the tiles be larger; the (tile, slices) with the fewest
// bytes per workgroup among those that run at once. At most four slices of at
// least 1024 (measured, FFN value, us, best whole / best cut: 0.4B 64 rows 11.1 /
// 7.8, 128 rows 11.0 / 8.7; 1.5B 64 rows 19.6 / 14.6, and 14.2 with eight slices,
// less than their extra partials cost the LayerNorm), and only up to 256 rows.
// Beyond, the partials that the LayerNorm reads grow with the rows and the gain
// depends on the shape (whole prefills, us, whole / cut: 0.4B 261 rows 2387 /
// 2283, 300 2442 / 2449, 400 2578 / 2607, 512 2831 / 2893; 0.1B 480 rows 1206 /
// 1226; 1.5B 257 rows 4592 / 4273, 512 5579 / 5335): one line for all leaves 4 to
// 7 % of the 1.5B shape there, until the plan counts the partials' bytes.
static int frag_plan(int M, int N, int K, int cus, int *splits) {
  GemmProb p = {};
  p.N = N;
  int best = frag_tile(&p, 1, M, cus);
  *splits = 1;
  if (M > 256) return best;
  int64_t bytes = INT64_MAX;
  for (int i = 0; i < kFragOneRound; ++i) {
    for (int s = 1; s <= 4 && K / s >= 1024; s *= 2) {
      if (frag_units(kFragTiles[i], M, N) * s > cus) break;
      const int64_t b = (int64_t)(4 * kFragTiles[i].bm + 2 * kFragTiles[i].bn) * ((K + s - 1) / s);
      if (b < bytes) {
        bytes = b;
        best = i;
        *splits = s;
      }
    }
  }
  return best;
}

int gemm_frag_splits(int M, int N, int K) {
  int s;
  frag_plan(M, N, K, mk_cus() > 0 ? mk_cus() : 256, &s);
  return s;
}

int launch_gemm_frag(const GemmProb *probs, int nprob, int M, hipStream_t st, int splits, int64_t part_stride) {
  if (nprob < 1 || nprob > kFragProbs || M <= 0 || splits < 1 || (splits & (splits - 1))) return RWKV7_ESHAPE;
  if (splits > 1 && (nprob != 1 || probs[0].epi != GEPI_F32)) return RWKV7_EINVAL;
  const int cus = mk_cus() > 0 ? mk_cus() : 256;
  for (int i = 0; i < nprob; ++i) {
    const GemmProb &p = probs[i];
    if (!p.A || !p.Wf || !p.Y) return RWKV7_EINVAL;
    if (p.N <= 0 || p.K <= 0 || p.nksf != (p.K + 31) / 32 || p.bf != probs[0].bf) return RWKV7_ESHAPE;
    if (p.epi == GEPI_ADD_F32 && (p.N % 4 || p.ldy % 4)) return RWKV7_ESHAPE;
  }
  int planned = 1;
  const int ti = splits > 1 ? frag_plan(M, probs[0].N, probs[0].K, cus, &planned) : frag_tile(probs, nprob, M, cus);
  if (splits > 1 && planned != splits) return RWKV7_EINVAL;
  const FragTile t = kFragTiles[ti];
  FragGroup g;
  g.nprob = nprob;
  g.M = M;
  g.m_tiles = (M + t.bm - 1) / t.bm;
  g.splits = splits;
  g.part_stride = part_stride;
  int64_t units = 0;
  for (int i = 0; i < kFragProbs; ++i) {
    g.unit_begin[i] = (int)units;
    g.p[i] = probs[i < nprob ? i : 0];
    if (i < nprob) units += (int64_t)((probs[i].N + t.bn - 1) / t.bn) * splits;
  }
  const int64_t items = units * g.m_tiles;
  if (items > INT32_MAX - 8) return RWKV7_ESHAPE;
  g.items = (int)items;
  g.per_xcd = (int)((items + 7) / 8);
  const bool bf = probs[0].bf != 0, ring = items <= cus && frag_ring(probs, nprob, M, kFragRingMinK);
  const dim3 grid(8u * (unsigned)g.per_xcd);
#define RWKV7_FRAG(...)                                                            \
  if (bf) gemm_frag_kernel<__VA_ARGS__, true><<<grid, kFragThreads, 0, st>>>(g);   \
  else gemm_frag_kernel<__VA_ARGS__, false><<<grid, kFragThreads, 0, st>>>(g);     \
  break;
#define RWKV7_FRAG_RING(...)                                                              \
  {                                                                                       \
    if (bf) gemm_frag_ring_kernel<__VA_ARGS__, true><<<grid, kFragThreads, 0, st>>>(g);   \
    else gemm_frag_ring_kernel<__VA_ARGS__, false><<<grid, kFragThreads, 0, st>>>(g);     \
    break;                                                                                \
  }
  switch (ti) {
    case 0: RWKV7_FRAG(1, 2, 1, 1, 8, 2)
    case 1: RWKV7_FRAG(2, 2, 1, 1, 8, 2)
    case 2: RWKV7_FRAG(2, 4, 1, 1, 8, 1)
    case 3: RWKV7_FRAG(2, 4, 2, 1, 4, 1)
    case 4: RWKV7_FRAG(2, 4, 1, 2, 4, 1)
    case 5:
      if (ring) RWKV7_FRAG_RING(2, 4, 2, 2, 2, 4)
      RWKV7_FRAG(2, 4, 2, 2, 2, 1)
    default: RWKV7_FRAG_RING(4, 4, 2, 2, 2, 3)
  }
#undef RWKV7_FRAG
#undef RWKV7_FRAG_RING
  RWKV7_CHECK_LAUNCH();
  return RWKV7_OK;
}

}  // namespace rwkv7
