// Device-wide exclusive scan of 32-bit counts and a stable LSD radix sort of
// (32-bit key, 32-bit value) pairs, used by compaction, the lexicographic
// vertex sort and the Morton sort of the LBVH.
//
// Radix sort, one 8-bit digit per pass:
//   1. count:   each 1024-lane workgroup counts the digits of its tile;
//   2. scan:    an exclusive scan of hist[digit][tile] gives every (digit,
//               tile) its base.  With at most kFewTiles tiles there is no scan:
//               each workgroup of the scatter adds up hist[tile][digit] itself;
//   3. scatter: each wave ranks a contiguous part of the tile stably, round by
//               round (8-ballot digit match, its digit counts in LDS), the
//               counts are scanned over the waves once, and the keys are
//               written to base + rank.  Keys are moved once per pass.
#include "iso_internal.hpp"

namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

// block exclusive scan of one value per lane; returns the exclusive prefix and
// writes the block total to *total
template <int BLOCK>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *s_tmp, uint32_t *total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == 63) s_tmp[w] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < BLOCK / 64; ++k) {
    const uint32_t t = s_tmp[k];
    before += k < w ? t : 0u;
    all += t;
  }
  *total = all;
  __syncthreads();
  return before + inc - v;
}

// Short arrays in one launch: one workgroup, kSmallItems consecutive words per
// lane and step.  Three launches and the gaps between them take about 15 us;
// a step takes 2.
constexpr int kSmallItems = 16;
struct __attribute__((packed, aligned(4))) uint4u {
  uint32_t x, y, z, w;
};
constexpr int64_t kSmallScan = 4 * 1024 * kSmallItems;

__global__ __launch_bounds__(1024) void scan_small_kernel(const uint32_t *in, int n, uint32_t *out,
                                                          uint32_t *total) {
  __shared__ uint32_t s_tmp[1024 / 64];
  uint32_t carry = 0;
  for (int base = 0; base < n; base += 1024 * kSmallItems) {
    const int i0 = base + threadIdx.x * kSmallItems;
    const bool whole = i0 + kSmallItems <= n;
    union {
      uint32_t v[kSmallItems];
      uint4u q[kSmallItems / 4];
    };
    uint32_t sum = 0, tot;
    if (whole) {
#pragma unroll
      for (int k = 0; k < kSmallItems / 4; ++k) q[k] = *(const uint4u *)(in + i0 + 4 * k);
    } else {
#pragma unroll
      for (int k = 0; k < kSmallItems; ++k) v[k] = i0 + k < n ? in[i0 + k] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) sum += v[k];
    uint32_t ex = carry + block_excl_scan<1024>(sum, s_tmp, &tot);
#pragma unroll
    for (int k = 0; k < kSmallItems; ++k) {
      const uint32_t t = v[k];
      v[k] = ex;
      ex += t;
    }
    if (whole) {
#pragma unroll
      for (int k = 0; k < kSmallItems / 4; ++k) *(uint4u *)(out + i0 + 4 * k) = q[k];
    } else {
#pragma unroll
      for (int k = 0; k < kSmallItems; ++k)
        if (i0 + k < n) out[i0 + k] = v[k];
    }
    carry += tot;
  }
  if (threadIdx.x == 0 && total) *total = carry;
}

__global__ __launch_bounds__(kScanBlock) void scan_reduce_kernel(const uint32_t *in, int64_t n,
                                                                 uint32_t *sums) {
  __shared__ uint32_t s_tmp[kScanBlock / 64];
  int64_t base = (int64_t)blockIdx.x * kScanTile;
  uint32_t v = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t i = base + (int64_t)k * kScanBlock + threadIdx.x;
    if (i < n) v += in[i];
  }
  uint32_t tot;
  block_excl_scan<kScanBlock>(v, s_tmp, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// single workgroup: exclusive scan of m block sums in place, total to *total
__global__ __launch_bounds__(1024) void scan_sums_kernel(uint32_t *sums, int64_t m,
                                                         uint32_t *total) {
  __shared__ uint32_t s_tmp[1024 / 64];
  __shared__ uint32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < m; base += 1024) {
    int64_t i = base + threadIdx.x;
    uint32_t v = i < m ? sums[i] : 0u;
    uint32_t tot;
    uint32_t ex = block_excl_scan<1024>(v, s_tmp, &tot);
    if (i < m) sums[i] = ex + s_carry;
    __syncthreads();
    if (threadIdx.x == 0) s_carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0 && total) *total = s_carry;
}

__global__ __launch_bounds__(kScanBlock) void scan_down_kernel(const uint32_t *in, int64_t n,
                                                               const uint32_t *sums,
                                                               uint32_t *out) {
  __shared__ uint32_t s_tmp[kScanBlock / 64];
  int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  uint32_t v[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t i = base + k;
    v[k] = i < n ? in[i] : 0u;
    s += v[k];
  }
  uint32_t tot;
  uint32_t ex = block_excl_scan<kScanBlock>(s, s_tmp, &tot) + sums[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t i = base + k;
    if (i < n) out[i] = ex;
    ex += v[k];
  }
}

// ---------------------------------------------------------------- radix sort
constexpr int kSortBlock = 1024;
constexpr int kSortWaves = kSortBlock / 64;

// For lane's digit d (8 bits), mask of lanes in the wave holding the same digit.
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    bool bit = (d >> b) & 1u;
    uint64_t bb = __ballot(bit && valid);
    m &= bit ? bb : ~bb;
  }
  return m;
}

// Tiles this few in number need no scan of the histograms between the
// count and the scatter: every scatter workgroup reads all of them (256 KB at
// most, from L2) instead of three launches.
constexpr int kFewTiles = 256;

// hist[tile][digit] if FEW, hist[digit][tile] else
template <int ITEMS, bool FEW>
__global__ __launch_bounds__(kSortBlock) void radix_count_kernel(const uint32_t *keys, int64_t n,
                                                                 int shift, uint32_t *hist,
                                                                 int ntiles) {
  __shared__ uint32_t s_cnt[256];
  if (threadIdx.x < 256) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  int64_t base = (int64_t)blockIdx.x * (kSortBlock * ITEMS);
  // every key requested before the first count (a load inside the counting
  // loop would wait for its value before the next one is issued)
  uint32_t keyv[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = base + (int64_t)k * kSortBlock + threadIdx.x;
    keyv[k] = i < n ? keys[i] : 0u;
  }
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = base + (int64_t)k * kSortBlock + threadIdx.x;
    // Lanes with the first lane's digit are added at once: neighbouring keys
    // often share their upper digits, and 64 adds to one word take 130 cycles.
    const uint32_t d = i < n ? (keyv[k] >> shift) & 255u : 256u;
    const uint32_t first = __builtin_amdgcn_readfirstlane(d);
    const uint64_t same = __ballot(d == first);
    if (first < 256u && (threadIdx.x & 63) == 0) atomicAdd(&s_cnt[first], (uint32_t)__popcll(same));
    if (d < 256u && d != first) atomicAdd(&s_cnt[d], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 256)
    hist[FEW ? (int64_t)blockIdx.x * 256 + threadIdx.x
             : (int64_t)threadIdx.x * ntiles + blockIdx.x] = s_cnt[threadIdx.x];
}

// Tile element order: wave w's part, ITEMS * 64 keys, round by round, lane by
// lane, so ranks are stable in global index order.  A wave counts its digits
// without a barrier; only the sums over the waves need the workgroup.
template <int ITEMS, bool FEW>
__global__ __launch_bounds__(kSortBlock) void radix_scatter_kernel(
    const uint32_t *keys, const uint32_t *vals, int64_t n, int shift, const uint32_t *hist,
    int ntiles, uint32_t *keys_out, uint32_t *vals_out) {
  __shared__ uint32_t s_wcnt[kSortWaves][256];  // per wave: digit counts, then bases
  // Whole tiles of several keys per digit are put in order in LDS and written
  // out from there: a store of 64 keys then covers a few runs instead of 64
  // lines, which the address unit takes one a cycle.
  constexpr bool kStaged = ITEMS >= 4;
  __shared__ uint32_t s_all[FEW ? 4 : 1][256], s_before[FEW ? 4 : 1][256], s_sum[4];
  __shared__ uint32_t s_first[256], s_to[256], s_tile[4];
  __shared__ uint32_t s_stage[kStaged ? kSortBlock * ITEMS : 1];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t base = (int64_t)blockIdx.x * (kSortBlock * ITEMS) + w * (64 * ITEMS);
  // the whole tile's keys are requested up front (and its values before the
  // keys go out), so one memory latency is exposed per tile instead of one per
  // round
  uint32_t keyv[ITEMS], valv[ITEMS], rank[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = base + k * 64 + lane;
    keyv[k] = i < n ? keys[i] : 0u;
    if (!kStaged) valv[k] = i < n ? vals[i] : 0u;
  }
  if (FEW) {  // all counts of each digit, and those in the tiles before this one
    const int d = tid & 255, g = tid >> 8;
    uint32_t all = 0, before = 0;
#pragma unroll 8
    for (int t = g; t < ntiles; t += 4) {
      const uint32_t c = hist[t * 256 + d];
      all += c;
      before += t < (int)blockIdx.x ? c : 0u;
    }
    s_all[g][d] = all;
    s_before[g][d] = before;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) s_wcnt[w][q * 64 + lane] = 0;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const bool valid = base + k * 64 + lane < n;
    const uint32_t d = (keyv[k] >> shift) & 255u;
    const uint64_t m = match_digit(d, valid);
    const uint32_t in_round = __builtin_amdgcn_mbcnt_hi(
        (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    const uint32_t had = s_wcnt[w][d];
    rank[k] = had + in_round;
    __builtin_amdgcn_wave_barrier();
    if (valid && in_round == 0) s_wcnt[w][d] = had + (uint32_t)__popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  uint32_t run = 0, mine = 0, all_inc = 0, tile_inc = 0;  // of digit tid
  if (tid < 256) {
    if (FEW) {
      const uint32_t all = s_all[0][tid] + s_all[1][tid] + s_all[2][tid] + s_all[3][tid];
      all_inc = wave_incl_scan(all);
      if (lane == 63) s_sum[w] = all_inc;
      run = all_inc - all + s_before[0][tid] + s_before[1][tid] + s_before[2][tid] + s_before[3][tid];
    } else {
      run = hist[(int64_t)tid * ntiles + blockIdx.x];
    }
    uint32_t c[kSortWaves];
#pragma unroll
    for (int q = 0; q < kSortWaves; ++q) c[q] = s_wcnt[q][tid];
#pragma unroll
    for (int q = 0; q < kSortWaves; ++q) {
      s_wcnt[q][tid] = mine;
      mine += c[q];
    }
    if (kStaged) {
      tile_inc = wave_incl_scan(mine);
      if (lane == 63) s_tile[w] = tile_inc;
    }
  }
  __syncthreads();
  if (tid < 256) {
    if (FEW)  // the digits of the waves before the digit's
      for (int q = 0; q < w; ++q) run += s_sum[q];
    uint32_t first = tile_inc - mine;  // the tile's keys of smaller digits
    if (kStaged)
      for (int q = 0; q < w; ++q) first += s_tile[q];
    s_first[tid] = first;
    s_to[tid] = run - first;
  }
  __syncthreads();
  if (!kStaged) {
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      if (base + k * 64 + lane >= n) break;
      const uint32_t d = (keyv[k] >> shift) & 255u;
      const uint32_t pos = s_first[d] + s_to[d] + s_wcnt[w][d] + rank[k];
      keys_out[pos] = keyv[k];
      vals_out[pos] = valv[k];
    }
    return;
  }
  // the tile in sorted order through LDS, keys then values
  const int64_t tile0 = (int64_t)blockIdx.x * (kSortBlock * ITEMS);
  const int count = (int)min(n - tile0, (int64_t)(kSortBlock * ITEMS));
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const uint32_t d = (keyv[k] >> shift) & 255u;
    rank[k] += s_first[d] + s_wcnt[w][d];
    if (base + k * 64 + lane < n) s_stage[rank[k]] = keyv[k];
  }
#pragma unroll
  for (int k = 0; k < ITEMS; ++k)
    valv[k] = base + k * 64 + lane < n ? vals[base + k * 64 + lane] : 0u;
  __syncthreads();
  uint32_t to[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int i = k * kSortBlock + tid;
    if (i >= count) break;
    const uint32_t key = s_stage[i];
    to[k] = s_to[(key >> shift) & 255u] + i;
    keys_out[to[k]] = key;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ITEMS; ++k)
    if (base + k * 64 + lane < n) s_stage[rank[k]] = valv[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int i = k * kSortBlock + tid;
    if (i >= count) break;
    vals_out[to[k]] = s_stage[i];
  }
}

__global__ void iota_kernel(uint32_t *p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (uint32_t)i;
}

}  // namespace

namespace iso {

// out[i] = sum(in[0..i)); *d_total (device, may be null) = sum of all.
// tmp: workspace of at least scan_tmp_words(n) words.
size_t scan_tmp_words(int64_t n) { return (size_t)((n + kScanTile - 1) / kScanTile) + 1; }

int exclusive_scan_u32(iso_ctx *ctx, const uint32_t *d_in, uint32_t *d_out, int64_t n,
                       uint32_t *d_total, uint32_t *d_tmp) {
  if (n <= 0) return ISO_OK;
  if (n <= kSmallScan) {
    hipLaunchKernelGGL(scan_small_kernel, dim3(1), dim3(1024), 0, ctx->stream, d_in, (int)n, d_out,
                       d_total);
    ISO_HIP_CHECK(ctx, hipGetLastError());
    return ISO_OK;
  }
  int64_t nb = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(scan_reduce_kernel, dim3((unsigned)nb), dim3(kScanBlock), 0, ctx->stream,
                     d_in, n, d_tmp);
  hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(1024), 0, ctx->stream, d_tmp, nb, d_total);
  hipLaunchKernelGGL(scan_down_kernel, dim3((unsigned)nb), dim3(kScanBlock), 0, ctx->stream, d_in,
                     n, (const uint32_t *)d_tmp, d_out);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

int iota_u32(iso_ctx *ctx, uint32_t *d, int64_t n) {
  if (n <= 0) return ISO_OK;
  hipLaunchKernelGGL(iota_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, d,
                     n);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

// Stable sort of (key, val) by the low `bits` bits of key.  Buffers a/b are
// ping-ponged; the sorted result ends in (*keys, *vals) which point to one of
// the two buffer pairs on return.
int radix_sort_pairs(iso_ctx *ctx, uint32_t **keys, uint32_t **vals, uint32_t *keys_alt,
                     uint32_t *vals_alt, int64_t n, int bits) {
  if (n <= 1) return ISO_OK;
  // keys per tile = 1024 lanes x items.  As many tiles as there are CUs while
  // the keys last (a few large tiles leave most of the chip idle: 160,000 keys
  // in 10 tiles took 50 us a pass with its counts and scan, in 160 tiles 9 us),
  // then 16 items: fewer histograms to scan and one exposed load latency per 16K
  // keys.  ISO_SORT_ITEMS=4 or 8 in the environment selects those tiles.
  int items = 1;
  while (items < 16 && n > (int64_t)kFewTiles * kSortBlock * items) items *= 2;
  if (const char *e = std::getenv("ISO_SORT_ITEMS")) {
    const int v = std::atoi(e);
    if (v == 4 || v == 8) items = v;
  }
  const int64_t tile = (int64_t)kSortBlock * items;
  int ntiles = (int)((n + tile - 1) / tile);
  const bool few = ntiles <= kFewTiles;
  size_t hwords = (size_t)256 * ntiles;
  void *hist = nullptr, *tmp = nullptr;
  ISO_TRY(ws_get(ctx, WS_SORT_HIST, sizeof(uint32_t) * hwords, false, &hist));
  if (!few)
    ISO_TRY(ws_get(ctx, WS_SCAN_TMP, sizeof(uint32_t) * scan_tmp_words((int64_t)hwords), false, &tmp));
  uint32_t *ka = *keys, *va = *vals, *kb = keys_alt, *vb = vals_alt;
  for (int shift = 0; shift < bits; shift += 8) {
    auto launch = [&](auto count, auto scatter) {
      hipLaunchKernelGGL(count, dim3(ntiles), dim3(kSortBlock), 0, ctx->stream, ka, n, shift,
                         (uint32_t *)hist, ntiles);
      if (!few)
        ISO_TRY(exclusive_scan_u32(ctx, (uint32_t *)hist, (uint32_t *)hist, (int64_t)hwords,
                                   nullptr, (uint32_t *)tmp));
      hipLaunchKernelGGL(scatter, dim3(ntiles), dim3(kSortBlock), 0, ctx->stream, ka, va, n, shift,
                         (const uint32_t *)hist, ntiles, kb, vb);
      return ISO_OK;
    };
    if (few) {
      switch (items) {
        case 1: ISO_TRY(launch(radix_count_kernel<1, true>, radix_scatter_kernel<1, true>)); break;
        case 2: ISO_TRY(launch(radix_count_kernel<2, true>, radix_scatter_kernel<2, true>)); break;
        case 4: ISO_TRY(launch(radix_count_kernel<4, true>, radix_scatter_kernel<4, true>)); break;
        case 8: ISO_TRY(launch(radix_count_kernel<8, true>, radix_scatter_kernel<8, true>)); break;
        default: ISO_TRY(launch(radix_count_kernel<16, true>, radix_scatter_kernel<16, true>));
      }
    } else if (items == 16) {
      ISO_TRY(launch(radix_count_kernel<16, false>, radix_scatter_kernel<16, false>));
    } else if (items == 8) {
      ISO_TRY(launch(radix_count_kernel<8, false>, radix_scatter_kernel<8, false>));
    } else {
      ISO_TRY(launch(radix_count_kernel<4, false>, radix_scatter_kernel<4, false>));
    }
    ISO_HIP_CHECK(ctx, hipGetLastError());
    uint32_t *t = ka; ka = kb; kb = t;
    t = va; va = vb; vb = t;
  }
  *keys = ka;
  *vals = va;
  return ISO_OK;
}

}  // namespace iso

// ---------------------------------------------------------------- vertex sort
namespace {

__global__ void key_from_xyz_kernel(const float *xyz, const uint32_t *idx, int64_t n, int comp,
                                    uint32_t *key) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) key[i] = __float_as_uint(xyz[3 * (int64_t)idx[i] + comp]);
}

__global__ void gather_xyz_kernel(const float *xyz, const uint32_t *idx, int64_t n, float *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    int64_t s = 3 * (int64_t)idx[i];
    out[3 * i] = xyz[s];
    out[3 * i + 1] = xyz[s + 1];
    out[3 * i + 2] = xyz[s + 2];
  }
}

// A marching-cubes vertex has at most one coordinate c that is not whole, so
// whole parts (bx, by, bz bits) and one fraction (its float bits, below 2^30)
// hold it exactly.  Within a whole x, a fraction of 0 comes before any other,
// and y decides among those; so these keys order as (x, y, z):
//   x | 1 | fraction of x | y | z | 0
//   x | 0 | y | 1 | fraction of y | z
//   x | 0 | y | 0 | z | fraction of z
struct LexBits {
  int bx, by, bz;
  __host__ __device__ int total() const { return bx + by + bz + 32; }
};

__device__ __forceinline__ void lex_decode(uint64_t key, LexBits b, float &x, float &y, float &z) {
  auto take = [&](int &at, int bits) {
    at -= bits;
    return (uint32_t)((key >> at) & ((1ull << bits) - 1));
  };
  int at = b.total();
  x = (float)take(at, b.bx);
  if (take(at, 1)) {
    x += __uint_as_float(take(at, 30));
    y = (float)take(at, b.by);
    z = (float)take(at, b.bz);
  } else {
    y = (float)take(at, b.by);
    if (take(at, 1)) {
      y += __uint_as_float(take(at, 30));
      z = (float)take(at, b.bz);
    } else {
      z = (float)take(at, b.bz);
      z += __uint_as_float(take(at, 30));
    }
  }
}

// *odd counts the vertices that their key does not give back bit for bit
__global__ void lex_encode_kernel(const float *xyz, int64_t n, LexBits b, uint32_t *lo,
                                  uint32_t *hi, uint32_t *odd) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float v[3] = {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]};
  const int bits[3] = {b.bx, b.by, b.bz};
  uint64_t whole[3];
  uint32_t frac[3];
  bool ok = true;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    ok = ok && v[c] >= 0.0f && v[c] < (float)(1u << bits[c]);
    const float w = ok ? floorf(v[c]) : 0.0f;
    whole[c] = (uint64_t)w;
    frac[c] = __float_as_uint(ok ? v[c] - w : 0.0f);
  }
  uint64_t key = whole[0] << (b.by + b.bz + 32);
  if (frac[0])
    key |= 1ull << (b.by + b.bz + 31) | (uint64_t)frac[0] << (b.by + b.bz + 1) |
           whole[1] << (b.bz + 1) | whole[2] << 1;
  else if (frac[1])
    key |= whole[1] << (b.bz + 31) | 1ull << (b.bz + 30) | (uint64_t)frac[1] << b.bz | whole[2];
  else
    key |= whole[1] << (b.bz + 31) | whole[2] << 30 | frac[2];
  float x, y, z;
  lex_decode(key, b, x, y, z);
  ok = ok && __float_as_uint(x) == __float_as_uint(v[0]) &&
       __float_as_uint(y) == __float_as_uint(v[1]) && __float_as_uint(z) == __float_as_uint(v[2]);
  if (!ok) atomicAdd(odd, 1u);
  lo[i] = (uint32_t)key;
  hi[i] = (uint32_t)(key >> 32);
}

__global__ void lex_decode_kernel(const uint32_t *lo, const uint32_t *hi, int64_t n, LexBits b,
                                  const uint32_t *odd, float *xyz) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || *odd) return;
  float x, y, z;
  lex_decode((uint64_t)hi[i] << 32 | lo[i], b, x, y, z);
  xyz[3 * i] = x;
  xyz[3 * i + 1] = y;
  xyz[3 * i + 2] = z;
}

__global__ void copy_f32_kernel(const float *src, float *dst, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

}  // namespace

namespace iso {

// Sorts n xyz triples lexicographically (x, then y, then z), in place, as the
// reference's thrust::sort over vec4f does (utils/typeOperation.h:1268-1279).
// Coordinates are non-negative, so float order equals the order of their bits;
// three stable LSD passes (z, y, x) of a 32-bit radix sort give the order.
int sort_triples_lex(iso_ctx *ctx, float *d_xyz, int64_t n) {
  if (n <= 1) return ISO_OK;
  void *ka, *kb, *va, *vb, *tmp;
  ISO_TRY(ws_get(ctx, WS_MC_KEYS_A, 4 * (size_t)n, false, &ka));
  ISO_TRY(ws_get(ctx, WS_MC_KEYS_B, 4 * (size_t)n, false, &kb));
  ISO_TRY(ws_get(ctx, WS_DF_IDX_A, 4 * (size_t)n, false, &va));
  ISO_TRY(ws_get(ctx, WS_DF_IDX_B, 4 * (size_t)n, false, &vb));
  ISO_TRY(ws_get(ctx, WS_MC_TMP, 12 * (size_t)n, false, &tmp));
  const unsigned g = (unsigned)((n + 255) / 256);
  uint32_t *idx = (uint32_t *)va, *idx_alt = (uint32_t *)vb;
  ISO_TRY(iota_u32(ctx, idx, n));
  for (int comp = 2; comp >= 0; --comp) {
    uint32_t *keys = (uint32_t *)ka;
    hipLaunchKernelGGL(key_from_xyz_kernel, dim3(g), dim3(256), 0, ctx->stream, d_xyz, idx, n, comp,
                       keys);
    uint32_t *k0 = keys, *v0 = idx;
    uint32_t *kalt = (uint32_t *)kb, *valt = idx_alt;
    ISO_TRY(radix_sort_pairs(ctx, &k0, &v0, kalt, valt, n, 32));
    // 4 passes: the result is back in the original buffers
    idx = v0;
    idx_alt = (v0 == (uint32_t *)va) ? (uint32_t *)vb : (uint32_t *)va;
  }
  hipLaunchKernelGGL(gather_xyz_kernel, dim3(g), dim3(256), 0, ctx->stream, d_xyz, idx, n,
                     (float *)tmp);
  hipLaunchKernelGGL(copy_f32_kernel, dim3((unsigned)((3 * n + 255) / 256)), dim3(256), 0,
                     ctx->stream, (const float *)tmp, d_xyz, 3 * n);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

// The same for the vertices of a grid of at most gx x gy x gz points with 64-bit
// keys: 8 passes or fewer where three 32-bit sorts take 12 and gather the
// coordinates in between (1.04M vertices of a 600x248x248 volume: three sorts 660
// us with tiles of 16K keys, 325 with these; the keys 210, and 170 since a tile is
// put in order in LDS).  Where a key would need more than 64 bits, and for vertices
// that no key holds (those of volumes with NaN or infinite samples), it falls back on
// the triples: *d_odd must be 0 on entry; the stream is synchronised.
int sort_vertices_lex(iso_ctx *ctx, float *d_xyz, int64_t n, int gx, int gy, int gz,
                      uint32_t *d_odd) {
  if (n <= 1) return ISO_OK;
  const LexBits b{ceil_log2((uint64_t)gx + 1), ceil_log2((uint64_t)gy + 1),
                  ceil_log2((uint64_t)gz + 1)};
  if (b.total() > 64) return sort_triples_lex(ctx, d_xyz, n);
  void *ka, *kb, *va, *vb, *pin;
  ISO_TRY(ws_get(ctx, WS_MC_KEYS_A, 4 * (size_t)n, false, &ka));
  ISO_TRY(ws_get(ctx, WS_MC_KEYS_B, 4 * (size_t)n, false, &kb));
  ISO_TRY(ws_get(ctx, WS_DF_IDX_A, 4 * (size_t)n, false, &va));
  ISO_TRY(ws_get(ctx, WS_DF_IDX_B, 4 * (size_t)n, false, &vb));
  ISO_TRY(pinned_get(ctx, 16, &pin));
  const unsigned g = (unsigned)((n + 255) / 256);
  uint32_t *lo = (uint32_t *)ka, *lo_alt = (uint32_t *)kb;
  uint32_t *hi = (uint32_t *)va, *hi_alt = (uint32_t *)vb;
  hipLaunchKernelGGL(lex_encode_kernel, dim3(g), dim3(256), 0, ctx->stream, d_xyz, n, b, lo, hi,
                     d_odd);
  auto sort = [&](uint32_t *&key, uint32_t *&key_alt, uint32_t *&val, uint32_t *&val_alt, int bits) {
    uint32_t *const k0 = key, *const v0 = val;
    ISO_TRY(radix_sort_pairs(ctx, &key, &val, key_alt, val_alt, n, bits));
    if (key != k0) key_alt = k0;
    if (val != v0) val_alt = v0;
    return ISO_OK;
  };
  ISO_TRY(sort(lo, lo_alt, hi, hi_alt, 32));
  ISO_TRY(sort(hi, hi_alt, lo, lo_alt, b.total() - 32));
  hipLaunchKernelGGL(lex_decode_kernel, dim3(g), dim3(256), 0, ctx->stream, (const uint32_t *)lo,
                     (const uint32_t *)hi, n, b, (const uint32_t *)d_odd, d_xyz);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(pin, d_odd, 4, hipMemcpyDeviceToHost, ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return *(const uint32_t *)pin ? sort_triples_lex(ctx, d_xyz, n) : ISO_OK;
}

}  // namespace iso
