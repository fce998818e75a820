// Normalised mutual information in the reference's float order, evaluated by
// a histogram workgroup once its pair's joint counts are complete.
//
// Reference: calculateMutualInformation (isosurfaces_cuda/src/JointHistogram.cu:
// 24-60), run per ordered pair (i, j) on the device:
//   hXY -= c * logf(c) over the nonzero bins, rows outer, columns inner;
//   hX  -= c * logf(c) over colSums[0..H), hY likewise over rowSums;
//   h = h / N + logf(N);  NMI = 2 (hX + hY - hXY) / (hX + hY), NaN -> 0.
// Each `-=` is one fused multiply-add (nvcc contracts a - b*c), so every
// accumulator is a chain of fmaf roundings in a fixed order; the result
// depends on that order and on nothing else.  The map entry (j, i) of the
// same unordered pair comes from the transposed histogram: its hXY chain
// visits the bins column by column, and its hX, hY are this pair's hY, hX
// (their sum is the same float).
//
// The chains are serial, so they are folded where many run side by side: the
// histogram workgroup only writes a pair's nonzero counts out in both chain
// orders, with the marginals, and fold_kernel (iso_hist.hip, iso_batch.hip)
// folds the chains of all pairs of a launch, eight to a wave.  Folded by four
// lanes of the histogram workgroup, the chains of 3,000 to 6,000 bins that
// 128-bin maps have kept a whole CU waiting.
//
// A pair's counts lie over the workgroup's lanes as the histogram's rows do (a
// wave has 16 or 8 consecutive rows, a lane 4 or 2 columns of them), so a bin's
// place in row-major order is the number of bins in the rows before plus a
// ballot prefix in its row, and in column-major order the number in the columns
// before plus those in the rows above: a prefix over the waves, then counted up
// row by row.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "iso_bins.hpp"
#include "iso_internal.hpp"

namespace iso {

// logf, correctly rounded for the counts it is applied to: the double
// logarithm of the value, rounded once to float.  For every integer from 1
// to 16,200,281 the exact logarithm lies at least 2^-48 (relative) away from
// a float rounding boundary (checked exhaustively on the CPU), far more than
// the error of a double logarithm, so any double log rounds to the one
// correct float.  Counts and field sizes stay below that bound unless a
// field has more than 16.2 million samples.
__device__ __forceinline__ float logf_cr(float x) { return (float)log((double)x); }

// Where a launch leaves what the chains need, per pair task: a header (number
// of nonzero bins, number of entries in `large`), the low 16 bits of the counts
// row by row and, list_bytes after it, column by column, those counts that need
// more in full (place, past 2^31 in the column list; count), and the marginals (H
// column sums, then H row sums).
struct ChainBufs {
  uint2 *head = nullptr;
  unsigned char *lists = nullptr;  // 2 * list_bytes per task
  size_t list_bytes = 0;           // a multiple of 16
  uint2 *large = nullptr;          // nlarge per task
  uint32_t nlarge = 0;
  uint32_t *marg = nullptr;        // 2 * H words per task
  const float *logs = nullptr;     // logf of 0 (taken as 0) to kLogs - 1
};
constexpr int kLogs = 65536;

// Room for one list: every nonzero bin, at most one per voxel, 16 bits each.
__host__ __device__ inline size_t chain_list_bytes(int H, int64_t F) {
  const int64_t n = (int64_t)H * H < F ? (int64_t)H * H : F;
  return ((size_t)n * 2 + 15) & ~(size_t)15;
}

// Counts of 2^16 and more, in both lists: at most one per 2^16 voxels and list.
__host__ __device__ inline size_t chain_large(int64_t F) { return 2 * (size_t)(F >> 16); }

// Takes a launch's ChainBufs out of p (chain_task_bytes per task + kChainPad).
inline void chain_carve(ChainBufs &b, void *p, int64_t ntasks, int H, int64_t F) {
  auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
  char *q = (char *)p;
  b.head = (uint2 *)q;
  q += up(sizeof(uint2) * (size_t)ntasks);
  b.marg = (uint32_t *)q;
  q += up(2 * sizeof(uint32_t) * (size_t)H * (size_t)ntasks);
  b.large = (uint2 *)q;
  b.nlarge = (uint32_t)chain_large(F);
  q += up(sizeof(uint2) * b.nlarge * (size_t)ntasks);
  b.lists = (unsigned char *)q;
  b.list_bytes = chain_list_bytes(H, F);
}

// Device bytes of ChainBufs per task (without the logarithms), and what rounding
// its parts up takes.
constexpr size_t kChainPad = 768;
__host__ __device__ inline size_t chain_task_bytes(int H, int64_t F) {
  return sizeof(uint2) * (1 + chain_large(F)) + 2 * chain_list_bytes(H, F) +
         2 * sizeof(uint32_t) * (size_t)H;
}

// number of set bits of m in the lanes below this one
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// LDS the NMI uses beside the histogram: nonzero bins per wave and column (then
// those in the waves before), nonzero bins in the rows (columns) before, the
// marginals and, for the double form, a list of nonzero bins (row << 8 | column):
// as many as fit one workgroup per CU (16-bit counters) or two.
template <bool PACK16>
struct PairLds {
  static constexpr int kH = PACK16 ? 256 : 128;    // most bins per axis
  static constexpr int kRows = kH / kHistWaves;    // rows of a wave
  static constexpr int kCols = kH / 64;            // columns of a lane
  static constexpr int kBins = PACK16 ? 10240 : 4608;  // most listed bins
  union {
    uint8_t colpre[kHistWaves][kH];
    uint16_t bins[kBins];
  };
  uint32_t rowbase[kH], colbase[kH];
  uint32_t rows[kH], cols[kH];
  uint32_t big, large;
  uint32_t wtot[kHistWaves];
};

// Clears the marginals and counters; a barrier comes before their use.
template <bool PACK16>
__device__ __forceinline__ void clear_pair_lds(PairLds<PACK16> &s) {
  if (threadIdx.x < PairLds<PACK16>::kH) s.rows[threadIdx.x] = s.cols[threadIdx.x] = 0u;
  if (threadIdx.x == 0) s.big = s.large = 0u;
}

// The count of bin (i, j): from the LDS histogram or, when gh is not null, from
// the H x H counts there (read past this CU's cache: atomics put them there).
template <bool PACK16>
__device__ __forceinline__ uint32_t pair_count(const uint32_t *s_hist, const uint32_t *gh, int H,
                                               int i, int j) {
  if (gh) return __hip_atomic_load(&gh[i * H + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return lds_count<PACK16>(s_hist, i, j);
}

// Bins of a lane in a row: two words of the LDS histogram.
template <bool PACK16>
constexpr int kSlotBins = PACK16 ? 4 : 2;

// Slot k of the histogram is words 2 (k % 64) and + 1 of row k / 64; lane t of
// the workgroup has slots t + 1024 q, q < kSlots.
template <bool PACK16>
constexpr int kSlots = PairLds<PACK16>::kH * 64 / kHistBlock;

template <bool PACK16>
__device__ __forceinline__ uint2 slot_words(const uint32_t *s_hist, int row, int l) {
  return reinterpret_cast<const uint2 *>(s_hist)[row * (kRowWords<PACK16> / 2) + l];
}

template <bool PACK16>
__device__ __forceinline__ uint32_t slot_count(uint2 v, int c) {
  if (PACK16) return ((c < 2 ? v.x : v.y) >> (16 * (c & 1))) & 0xffffu;
  return c == 0 ? v.x : v.y;
}

// Lists the nonzero bins of the LDS histogram (or of gh) if they are kBins at
// most, and returns their number (uniform).  Their order hangs on the counts
// alone: lane after lane, each its slots in turn.
template <bool PACK16>
__device__ __attribute__((always_inline)) uint32_t list_bins(const uint32_t *s_hist,
                                                             const uint32_t *gh, int H,
                                                             PairLds<PACK16> &s) {
  using L = PairLds<PACK16>;
  constexpr int kPer = kSlotBins<PACK16>;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  // kPer bits per slot of the lane: which of its bins are not zero
  uint64_t nz = 0ull;
#pragma unroll
  for (int q = 0; q < kSlots<PACK16>; ++q) {
    const int k = q * kHistBlock + (int)threadIdx.x;
    if (k >= H * 64) break;
    uint2 v = make_uint2(0u, 0u);
    if (!gh) v = slot_words<PACK16>(s_hist, k >> 6, k & 63);
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      const int j = (k & 63) * kPer + c;
      const uint32_t n = !gh ? slot_count<PACK16>(v, c)
                         : j < H ? pair_count<PACK16>(s_hist, gh, H, k >> 6, j) : 0u;
      nz |= (uint64_t)(n != 0u) << (kPer * q + c);
    }
  }
  // the lane's place in the wave's run, then the wave's in the list
  const uint32_t n = (uint32_t)__popcll(nz);
  uint32_t incl = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o, 64);
    if (l >= o) incl += t;
  }
  if (l == 63) s.wtot[w] = incl;
  __syncthreads();
  uint32_t at = incl - n, all = 0u;
#pragma unroll
  for (int q = 0; q < kHistWaves; ++q) {
    const uint32_t t = s.wtot[q];
    at += q < w ? t : 0u;
    all += t;
  }
  all = __builtin_amdgcn_readfirstlane(all);
  if (all > (uint32_t)L::kBins) return all;
  while (nz) {
    const int b = __ffsll((unsigned long long)nz) - 1;
    nz &= nz - 1ull;
    const int k = (b / kPer) * kHistBlock + (int)threadIdx.x;
    s.bins[at++] = (uint16_t)((k >> 6) << 8 | ((k & 63) * kPer + b % kPer));
  }
  __syncthreads();
  return all;
}

// f(i, j, count) for every nonzero bin of a pair whose bins are not listed: bin i
// H + j is lane (i H + j) % 1024's.
template <bool PACK16, class F>
__device__ __forceinline__ void each_bin(const uint32_t *s_hist, const uint32_t *gh, int H, F f) {
  const int di = kHistBlock / H, dj = kHistBlock - di * H;
  int i = (int)threadIdx.x / H, j = (int)threadIdx.x - i * H;
  while (i < H) {
    const uint32_t v = pair_count<PACK16>(s_hist, gh, H, i, j);
    if (v) f(i, j, v);
    i += di;
    j += dj;
    if (j >= H) {
      j -= H;
      ++i;
    }
  }
}

// Writes a pair's chain inputs out (task t of b).  The joint counts are in the
// LDS histogram (hist_bytes of it, overwritten) or, with GH, in gh (H x H 32-bit
// counts, set back to zero here).  s.rows and s.cols are zero and are left
// holding the marginals.  mirror: the column-by-column list is wanted too.
// Called by every lane of a 1024-lane workgroup with uniform arguments, after a
// barrier.
//
// The counts wait in registers while their LDS takes the lists, so the lists
// leave in coalesced stores (scattered 2-byte stores of some 4,000 bins to both
// lists would cost the L2 8,000 transactions per pair).  Counts past 16 bits
// (rare) go out one by one as well.
template <bool PACK16, bool GH>
__device__ __attribute__((always_inline)) void emit_chains(uint32_t *s_hist, int hist_bytes,
                                                           uint32_t *gh, int H, bool mirror,
                                                           PairLds<PACK16> &s, const ChainBufs &b,
                                                           int64_t t) {
  using L = PairLds<PACK16>;
  constexpr int kH = L::kH, R = L::kRows, C = L::kCols;
  constexpr int kLogR = PACK16 ? 4 : 3;
  int tid = threadIdx.x;
  // the lane id made opaque: inside a persistent task loop, addresses derived
  // from it must not be hoisted out of the loop (they would stay live across
  // the histogram phase and spill)
  asm volatile("" : "+v"(tid));
  const int l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = R * w, j0 = C * l;  // the lane's bins: rows i0 + r, columns j0 + c
  uint2 slot[R];                     // the lane's two words of each row
#pragma unroll
  for (int r = 0; r < R; ++r) {
    slot[r] = make_uint2(0u, 0u);
    if (!GH && i0 + r < H) slot[r] = slot_words<PACK16>(s_hist, i0 + r, l);
  }
  auto count = [&](int r, int c) -> uint32_t {
    if (GH)
      return i0 + r < H && j0 + c < H ? pair_count<PACK16>(nullptr, gh, H, i0 + r, j0 + c) : 0u;
    if (PACK16) return ((c < 2 ? slot[r].x : slot[r].y) >> (16 * (c & 1))) & 0xffffu;
    return c == 0 ? slot[r].x : slot[r].y;
  };
  uint32_t csum[C], cnz[C], rsum[R], all = 0u;
#pragma unroll
  for (int c = 0; c < C; ++c) csum[c] = cnz[c] = 0u;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    uint32_t rs = 0u, n = 0u;
    if (i0 + r < H) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t v = count(r, c);
        csum[c] += v;
        cnz[c] += v != 0u;
        rs += v;
        all |= v;
        n += (uint32_t)__popcll(__ballot(v != 0u));
      }
    }
    rsum[r] = rs;
    if (l == 0) s.rowbase[i0 + r] = n;
  }
  if (__ballot(all > 0xffffu) && l == 0) s.big = 1u;
  // row sums over the wave's 64 lanes by halving exchanges: across lane bit 32,
  // 16, ... a lane keeps the half of its rows that the bit selects and adds its
  // partner's copy of that half (R - 1 shuffles), then the low lane bits are
  // summed; lane l ends with row l >> (6 - kLogR)
#pragma unroll
  for (int st = 0; st < kLogR; ++st) {
    const int half = R >> (st + 1), sbit = 32 >> st;
    const bool up = (l & sbit) != 0;
#pragma unroll
    for (int k = 0; k < half; ++k) {
      const uint32_t give = up ? rsum[k] : rsum[half + k];
      const uint32_t keep = up ? rsum[half + k] : rsum[k];
      rsum[k] = keep + __shfl_xor(give, sbit, 64);
    }
  }
  uint32_t tot = rsum[0];
#pragma unroll
  for (int o = 32 >> kLogR; o > 0; o >>= 1) tot += __shfl_xor(tot, o, 64);
  if ((l & ((64 >> kLogR) - 1)) == 0) s.rows[i0 + (l >> (6 - kLogR))] = tot;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (csum[c]) atomicAdd(&s.cols[j0 + c], csum[c]);
    s.colpre[w][j0 + c] = (uint8_t)cnz[c];
  }
  __syncthreads();
  // column bases (waves 0-3) and row bases (waves 4-7); the marginals out
  uint32_t mine = 0u, incl = 0u;
  if (tid < 512) {
    const int q = tid & 255;
    if (q < kH) {
      if (tid < 256) {
#pragma unroll
        for (int v = 0; v < kHistWaves; ++v) {
          const uint32_t n = s.colpre[v][q];
          s.colpre[v][q] = (uint8_t)mine;  // at most 15 R
          mine += n;
        }
      } else {
        mine = s.rowbase[q];
      }
    }
    incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t u = __shfl_up(incl, o, 64);
      if (l >= o) incl += u;
    }
    if (l == 63) s.wtot[w] = incl;
  } else {
    const int q = tid & 255;
    if (q < H) b.marg[(2 * t + (tid < 768 ? 0 : 1)) * H + q] = tid < 768 ? s.cols[q] : s.rows[q];
  }
  __syncthreads();
  // (columns past H hold counts only for values past the interval given)
  const uint32_t nz = min(s.wtot[4] + s.wtot[5] + s.wtot[6] + s.wtot[7],
                          (uint32_t)(b.list_bytes / sizeof(uint16_t)));
  const bool wide = s.big != 0u;
  if (tid < 512) {
    uint32_t off = 0u;
    for (int q = tid < 256 ? 0 : 4; q < w; ++q) off += s.wtot[q];
    const int q = tid & 255;
    if (q < kH) (tid < 256 ? s.colbase : s.rowbase)[q] = incl - mine + off;
  }
  __syncthreads();
  unsigned char *la = b.lists + 2 * (size_t)t * b.list_bytes, *lb = la + b.list_bytes;
  // each list's room in LDS, whole 16-byte pieces
  const uint32_t room = (2u * nz + 15u) & ~15u;
  const bool staged = !GH && 2u * room <= (uint32_t)hist_bytes;
  uint16_t *wa = reinterpret_cast<uint16_t *>(s_hist), *wb = wa + room / 2;
  uint32_t col[C];  // the lane's columns' next places
#pragma unroll
  for (int c = 0; c < C; ++c) col[c] = s.colbase[j0 + c] + s.colpre[w][j0 + c];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (i0 + r >= H) continue;
    uint32_t v[C];
    uint64_t m[C];
    uint64_t any = 0ull;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      v[c] = count(r, c);
      m[c] = __ballot(v[c] != 0u);
      any |= m[c];
    }
    if (any == 0ull) continue;
    uint32_t row = s.rowbase[i0 + r];
#pragma unroll
    for (int c = 0; c < C; ++c) row += lanes_below(m[c]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (v[c]) {
        // places are permutations of [0, nz); the bounds only keep a wrong
        // count from writing past the lists
        if (staged) {
          if (row < nz) wa[row] = (uint16_t)v[c];
          if (mirror && col[c] < nz) wb[col[c]] = (uint16_t)v[c];
        } else {
          if (row < nz) reinterpret_cast<uint16_t *>(la)[row] = (uint16_t)v[c];
          if (mirror && col[c] < nz) reinterpret_cast<uint16_t *>(lb)[col[c]] = (uint16_t)v[c];
        }
        if (wide && v[c] > 0xffffu) {
          const uint32_t k = atomicAdd(&s.large, mirror ? 2u : 1u);
          uint2 *at = b.large + (size_t)t * b.nlarge + k;
          if (k < b.nlarge) at[0] = make_uint2(row, v[c]);
          if (mirror && k + 1u < b.nlarge) at[1] = make_uint2(col[c] | 1u << 31, v[c]);
        }
        if (GH) gh[(i0 + r) * H + j0 + c] = 0u;  // zero at rest (zero bins already are)
        ++row;
        ++col[c];
      }
    }
  }
  __syncthreads();
  if (tid == 0) b.head[t] = make_uint2(nz, min(s.large, b.nlarge));
  if (!staged) return;
  const uint4 *src = reinterpret_cast<const uint4 *>(s_hist);
  const int n16 = (int)(room / 16u);
  for (int k = tid; k < (mirror ? 2 : 1) * n16; k += kHistBlock)
    reinterpret_cast<uint4 *>(k < n16 ? la : lb)[k < n16 ? k : k - n16] = src[k];
}

// ---- the chains -------------------------------------------------------------
constexpr int kFoldPairs = 2;                // pairs of a workgroup
constexpr int kFoldChains = 4 * kFoldPairs;  // (i, j), (j, i), columns, rows of each
constexpr int kFoldBlock = 128;              // terms of a chain per step
constexpr int kFoldWaves = 5;                // the first folds, the others lay terms out
// terms of a chain's row in LDS, padded so that the chains' 16-byte reads meet
// different banks
constexpr int kFoldRow = kFoldBlock + 2;

struct FoldLds {
  alignas(16) float2 terms[2][kFoldChains][kFoldRow];
};

// Task t's outputs for fold_chains.
struct FoldOut {
  bool mirror;
  int64_t N;
  float *ij, *ji;
};

// The NMI of pair tasks t0 and t0 + 1 (below ntasks), by a workgroup of 5 waves.
// out(t) gives task t's outputs.
//
// Chain c of the 8 is pair c / 4's (i, j), (j, i), column or row chain.  Lane c
// of the first wave folds it, acc = fmaf(-c, logf(c), acc), in order, 128 terms
// a step from one of two LDS buffers, while each of the other waves lays the
// next 128 of a list out in the other; their counts are read three steps ahead and
// their logarithms looked up two steps ahead.  Past a chain's end the terms are
// (0, 0), and fmaf(-0, 0, acc) is acc exactly.
//
// The fold is a chain of dependent multiply-adds (about 0.6 us a step); by one
// wave alone, the counts, look-ups and stores between its folds took twice as
// long again.  Six such workgroups fit a CU; 256 terms a step and two waves for
// the four lists fit four, and two waves keep up with neither: 5,050 pairs of
// the 600x248x248 front (up to 9,400 terms) 90 -> 71 us, 32,896 pairs of 60,000
// voxels 741 -> 594, 2,016 of 128^3 fields 258 -> 247 (128 terms and two waves
// 98, 590, 410).
template <class Out>
__device__ __attribute__((always_inline)) void fold_chains(const ChainBufs &b, int H, int64_t t0,
                                                           int64_t ntasks, Out out, FoldLds &s) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // length of pair p's chain k (0 where there is none)
  auto length = [&](int p, int k) -> int {
    if (t0 + p >= ntasks) return 0;
    if (k >= 2) return H;
    if (k == 1 && !out(t0 + p).mirror) return 0;
    return __builtin_amdgcn_readfirstlane((int)b.head[t0 + p].x);
  };
  int most = H;
#pragma unroll
  for (int p = 0; p < kFoldPairs; ++p) most = max(most, length(p, 0));
  const int steps = (most + kFoldBlock - 1) / kFoldBlock;

  if (w == 0) {  // ---- the folds
    float acc = 0.0f;
    for (int q = 0; q < steps; ++q) {
      __syncthreads();
      if (lane < kFoldChains) {
        // 8 terms at a time, the next 8 on their way
        const float4 *row = reinterpret_cast<const float4 *>(s.terms[q & 1][lane]);
        constexpr int kQ = kFoldBlock / 32;
        float4 r0[kQ], r1[kQ];
        auto get = [&](float4(&r)[kQ], int k) {
#pragma unroll
          for (int u = 0; u < kQ; ++u) r[u] = row[k + u];
        };
        auto fold = [&](const float4(&r)[kQ]) {
#pragma unroll
          for (int u = 0; u < kQ; ++u) {
            acc = fmaf(-r[u].x, r[u].y, acc);
            acc = fmaf(-r[u].z, r[u].w, acc);
          }
        };
        get(r0, 0);
        for (int k = 0; k < kFoldBlock / 2; k += 2 * kQ) {
          get(r1, k + kQ);
          __builtin_amdgcn_sched_barrier(0);
          fold(r0);
          if (k + 2 * kQ < kFoldBlock / 2) get(r0, k + 2 * kQ);
          __builtin_amdgcn_sched_barrier(0);
          fold(r1);
        }
      }
    }
    // lanes 4 p .. 4 p + 3 hold pair p's chains
    const int p = (lane >> 2) & (kFoldPairs - 1);
    const float hji = __shfl(acc, 4 * p + 1, 64), hx = __shfl(acc, 4 * p + 2, 64),
                hy = __shfl(acc, 4 * p + 3, 64);
    if (lane < kFoldChains && (lane & 3) == 0 && t0 + p < ntasks) {
      const FoldOut o = out(t0 + p);
      const float fN = (float)o.N;
      const float lN = logf_cr(fN);
      const float fx = hx / fN + lN, fy = hy / fN + lN;
      const float sxy = fx + fy;
      float fxy = acc / fN + lN;
      float v = 2.0f * (sxy - fxy) / sxy;
      *o.ij = v != v ? 0.0f : v;
      if (o.mirror) {
        fxy = hji / fN + lN;
        v = 2.0f * (sxy - fxy) / sxy;
        *o.ji = v != v ? 0.0f : v;
      }
    }
    return;
  }

  // ---- the terms: wave w has list chains w - 1, w + 1, ... of the 4 (pair lc /
  // 2's row-major or column-major list) and, in the first step, the marginals'
  // chains of the same numbers
  constexpr int kLists = 2 * kFoldPairs, kOwn = (kLists + kFoldWaves - 2) / (kFoldWaves - 1);
  int len[kOwn];
  uint32_t nlarge[kOwn];
  const uint2 *large[kOwn];
  const unsigned char *src[kOwn];
#pragma unroll
  for (int u = 0; u < kOwn; ++u) {
    const int lc = w - 1 + u * (kFoldWaves - 1);
    len[u] = lc < kLists ? length(lc >> 1, lc & 1) : 0;
    const int64_t t = t0 + (len[u] ? lc >> 1 : 0);
    nlarge[u] = (uint32_t)__builtin_amdgcn_readfirstlane((int)b.head[t].y);
    large[u] = b.large + (size_t)t * b.nlarge;
    src[u] = b.lists + (2 * (size_t)t + (lc & 1)) * b.list_bytes;
  }
  constexpr int kPer = kFoldBlock / 64;  // terms of a chain a lane lays out per step
  static_assert(kPer == 2 || kPer == 4, "a load takes 2 or 4 counts");
  struct Counts {
    uint32_t v[kOwn][kPer];
  };
  // this lane's counts of step q: entries k .. k + kPer - 1 of each chain, k =
  // kFoldBlock q + kPer lane, 0 past the chain's end (a list's room is whole 16-byte
  // pieces, so those of its last entry can be read)
  auto load = [&](Counts &n, int q) {
#pragma unroll
    for (int u = 0; u < kOwn; ++u) {
#pragma unroll
      for (int c = 0; c < kPer; ++c) n.v[u][c] = 0u;
      if (q * kFoldBlock < len[u]) {
        const int k = q * kFoldBlock + kPer * lane, i = k < len[u] ? k : 0;
        uint32_t x[kPer];
        struct alignas(2 * kPer) Narrow { uint32_t v[kPer / 2]; };
        const Narrow y = reinterpret_cast<const Narrow *>(src[u])[i / kPer];
#pragma unroll
        for (int c = 0; c < kPer; c += 2) {
          x[c] = y.v[c / 2] & 0xffffu;
          x[c + 1] = y.v[c / 2] >> 16;
        }
        for (uint32_t e = 0; e < nlarge[u]; ++e) {
          const uint2 full = large[u][e];
          const uint32_t list = (uint32_t)(w - 1 + u * (kFoldWaves - 1)) & 1u;
#pragma unroll
          for (int c = 0; c < kPer; ++c)
            if (full.x == ((uint32_t)(k + c) | list << 31)) x[c] = full.y;
        }
#pragma unroll
        for (int c = 0; c < kPer; ++c) n.v[u][c] = k + c < len[u] ? x[c] : 0u;
      }
    }
  };
  struct Logs {
    float t[kOwn][kPer];
  };
  auto look_up = [&](const Counts &n, Logs &g, int q) {
#pragma unroll
    for (int u = 0; u < kOwn; ++u)
#pragma unroll
      for (int c = 0; c < kPer; ++c)
        g.t[u][c] = q * kFoldBlock < len[u] ? b.logs[min(n.v[u][c], (uint32_t)kLogs - 1u)] : 0.0f;
  };
  // rows past their chain's end are zeroed in both buffers and left
  auto put = [&](const Counts &n, Logs &g, int q) {
#pragma unroll
    for (int u = 0; u < kOwn; ++u) {
      const int lc = w - 1 + u * (kFoldWaves - 1);
      if (lc >= kLists || (q - 2) * kFoldBlock >= len[u]) continue;
      if (nlarge[u]) {  // counts past the table
#pragma unroll
        for (int c = 0; c < kPer; ++c)
          if (n.v[u][c] >= (uint32_t)kLogs) g.t[u][c] = logf_cr((float)n.v[u][c]);
      }
      float4 *row = reinterpret_cast<float4 *>(&s.terms[q & 1][4 * (lc >> 1) + (lc & 1)][kPer * lane]);
#pragma unroll
      for (int c = 0; c < kPer; c += 2)
        row[c / 2] = make_float4((float)n.v[u][c], g.t[u][c], (float)n.v[u][c + 1], g.t[u][c + 1]);
    }
  };
  auto log_of = [&](uint32_t v) -> float {
    float t = b.logs[min(v, (uint32_t)kLogs - 1u)];
    if (v >= (uint32_t)kLogs) t = logf_cr((float)v);
    return t;
  };
  // the marginals: kMarg steps (H <= 256), then zeros in both buffers
  constexpr int kMarg = 256 / kFoldBlock;
  auto put_marginals = [&](int q) {
#pragma unroll
    for (int u = 0; u < kOwn; ++u) {
      const int lc = w - 1 + u * (kFoldWaves - 1);
      if (lc >= kLists) continue;
      const int n = q < kMarg ? length(lc >> 1, 2 + (lc & 1)) : 0;
      const uint32_t *m = b.marg + (2 * (t0 + (n ? lc >> 1 : 0)) + (lc & 1)) * H;
#pragma unroll
      for (int c = 0; c < kPer; ++c) {
        const int i = 64 * c + lane, k = q * kFoldBlock + i;
        const uint32_t v = k < n ? m[k] : 0u;
        s.terms[q & 1][4 * (lc >> 1) + 2 + (lc & 1)][i] = make_float2((float)v, k < n ? log_of(v) : 0.0f);
      }
    }
  };
  Counts n0, n1, n2, n3;
  Logs g0, g1, g2;
  load(n0, 0);
  load(n1, 1);
  load(n2, 2);
  look_up(n0, g0, 0);
  look_up(n1, g1, 1);
  put(n0, g0, 0);
  put_marginals(0);
  for (int q = 0; q < steps; ++q) {
    __syncthreads();
    if (q + 1 < steps) {
      // n1, g1: step q + 1; n2: q + 2
      load(n3, q + 3);
      look_up(n2, g2, q + 2);
      put(n1, g1, q + 1);
      if (q < kMarg + 1) put_marginals(q + 1);
      n1 = n2;
      g1 = g2;
      n2 = n3;
    }
  }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// NMI of a pair in double from the exact counts (arguments as for emit_chains;
// the histogram's LDS is left as it is); the value is lane 0's, NaN included.
//
// Every lane sums the same bins in the same order whenever the counts are the
// same: bins that a counter drawn by the waves dealt out gave sums, and now and
// then a float, that changed from run to run.  With a bin per lane at most there
// is nothing to list (5,050 pairs of 5,000 voxels, 16 bins: 124 us listed, 115
// not; 64 bins, smooth fields: 151 listed, 175 not).  The list holds what the LDS
// has room for, and past it every bin is looked at (200 bins, noise of 4,700 bins:
// 1,064 us with room for 3,072, 431 with room for 10,240).
template <bool PACK16>
__device__ __attribute__((always_inline)) double nmi64_pair(const uint32_t *s_hist, uint32_t *gh,
                                                            int H, int64_t N, PairLds<PACK16> &s,
                                                            double (&s_red)[3][kHistWaves]) {
  using L = PairLds<PACK16>;
  const int tid = threadIdx.x;
  double sxy = 0.0, sx = 0.0, sy = 0.0;
  auto fold = [&](int i, int j, uint32_t c) {
    const double dc = (double)c;
    sxy += dc * log(dc);
    atomicAdd(&s.rows[i], c);
    atomicAdd(&s.cols[j], c);
    if (gh) gh[i * H + j] = 0u;  // zero at rest
  };
  const uint32_t nbins = __builtin_amdgcn_readfirstlane(H * H) > kHistBlock
                             ? list_bins<PACK16>(s_hist, gh, H, s)
                             : ~0u;
  if (nbins <= (uint32_t)L::kBins) {
    for (uint32_t k = tid; k < nbins; k += kHistBlock) {
      const int i = s.bins[k] >> 8, j = s.bins[k] & 255;
      fold(i, j, pair_count<PACK16>(s_hist, gh, H, i, j));
    }
  } else {
    each_bin<PACK16>(s_hist, gh, H, fold);
  }
  __syncthreads();
  if (tid < H) {
    const uint32_t r = s.rows[tid], c = s.cols[tid];
    if (r) sx = (double)r * log((double)r);
    if (c) sy = (double)c * log((double)c);
  }
  sxy = wave_sum(sxy);
  sx = wave_sum(sx);
  sy = wave_sum(sy);
  const int w = tid >> 6;
  if ((tid & 63) == 0) { s_red[0][w] = sxy; s_red[1][w] = sx; s_red[2][w] = sy; }
  __syncthreads();
  double v = 0.0;
  if (tid == 0) {
    double txy = 0, tx = 0, ty = 0;
    for (int k = 0; k < kHistWaves; ++k) { txy += s_red[0][k]; tx += s_red[1][k]; ty += s_red[2][k]; }
    const double dN = (double)N, lnN = log(dN);
    const double hx = lnN - tx / dN, hy = lnN - ty / dN, hxy = lnN - txy / dN;
    v = 2.0 * (hx + hy - hxy) / (hx + hy);
  }
  return v;
}

// logf of the counts 0 to kLogs - 1: the context's table, filled on
// first use, or into the caller's memory.
int nmi_logs(iso_ctx *ctx, const float **out);
int nmi_logs_fill(iso_ctx *ctx, float *d_logs);

// Tasks of a launch in the reference's float order, ntasks at most: as many whole
// rounds of workgroups as limit_mib MiB of the chains' inputs hold (F: the tasks'
// largest), one task in any case.  ISO_NMI_CHAIN_MIB in the environment sets another
// limit.  Every launch ends with its last pairs and its folds, so few large ones are
// better, until their inputs no longer stay in the caches.  One volume's pairs: 2
// GiB, 1 GiB up to 128 bins (600x248x248 front, 256 bins, by 2 GiB, 1 GiB, 512 MiB:
// 2.04, 2.13, 2.24 ms; 256 isovalues of 60,000 voxels, 128 bins: 1.89, 1.86, 1.92).
// A batch, whose pairs come from queues: 2 GiB, 512 MiB up to 128 bins (48 volumes,
// 186,551 pairs, 128 bins, by 2 GiB, 1 GiB, 512 MiB: 57.4, 55.7, 53.3 ms; 256 bins:
// 66.6, 68.8, 73.8).
int chain_tasks(const iso_ctx *ctx, int H, int64_t F, int64_t ntasks, int limit_mib);

// The context's ChainBufs for a launch of ntasks tasks.
int chain_get(iso_ctx *ctx, int64_t ntasks, int H, int64_t F, ChainBufs &b);

// Device buffers one launch of the histogram + NMI kernels works in: merged
// 32-bit histograms and slice arrival counters per task (zero at rest), the
// slices' own histograms (hist_parts_bytes; null: they are added to the merged
// ones) and, for the reference-order NMI, the chains' inputs.
struct HistBufs {
  uint32_t *ghist = nullptr;
  uint32_t *arrive = nullptr;
  uint32_t *parts = nullptr;
  ChainBufs chains;
};

// Bytes of HistBufs::parts for a launch over nt pairs (0: pairs are not cut up).
size_t hist_parts_bytes(const iso_ctx *ctx, int64_t F, int H, uint32_t flags, int64_t nt);

// One launch over tasks d_tasks[0, nt) with the caller's buffers; variant
// 0 or 1 is the kernel shape (the autotuner's two candidates).
int hist_launch(iso_ctx *ctx, const float *d_fields, int n, int64_t F, int H, int multi,
                uint32_t flags, const float *d_mins, const float *d_maxs, float *d_map,
                const int2 *d_tasks, int nt, uint32_t *d_joint, uint32_t *d_rows,
                uint32_t *d_cols, const HistBufs &b, int variant);

}  // namespace iso
