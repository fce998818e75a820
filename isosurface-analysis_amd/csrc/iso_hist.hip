// Joint histograms + normalised mutual information over pairs of distance
// fields, and per-field intervals.
//
// Reference semantics (isosurfaces_cuda/src/JointHistogram.cu):
//   pair (i,j): min = min(min_i,min_j), max = max(max_i,max_j),
//   step = (max-min)/H, bin(v) = (int)((v-min)/step) clamped to H-1, step==0 -> 0
//   (findBucket_d, :63-75; :127-129); hist[row*H+col], row from field i.
//   NMI = 2 (Hx+Hy-Hxy)/(Hx+Hy), NaN -> 0 (calculateMutualInformation, :24-60).
//
// MI355X design:
//   - one workgroup (1024 lanes, 16 waves) owns one unordered pair (or one
//     voxel slice of it when there are too few pairs to fill 256 CUs); the
//     pair's joint histogram is privatised in LDS (32-bit counters for
//     H <= 128: 68 KB; 16-bit counters packed two per dword for H <= 256:
//     128 KB of the 160 KB LDS), a row as long whatever H is;
//   - bins are computed exactly in fixed point, and 16-bit counters hand on
//     32,768 of their count before they can wrap (iso_bins.hpp);
//   - slices of one pair leave their LDS histograms in memory, and a kernel adds
//     them up into a global 32-bit histogram, which also takes what 16-bit
//     counters handed on; a pair's counts go back from there into LDS and the
//     zeros are restored, so the buffer is zero at rest;
//   - with ISO_COMPAT_NMI32 the NMI is the reference's float evaluation in the
//     reference's order: the workgroup writes the pair's nonzero counts out in
//     both chain orders and a second kernel folds the chains of all pairs
//     (iso_nmi.hpp); without it, the same quantity from the exact integer
//     counts in double (sum c ln c), in the same kernel;
//   - pairs come in tiles of 8 x 8 fields, each as two of 4 x 8, and workgroup
//     ids are remapped so that an XCD runs the pairs of a tile (two workgroups
//     per CU: 64 at a time, 16 fields) or half a tile (32, 12 fields) at a time,
//     which share their fields in its L2 (row by row, 33 fields for 32 pairs,
//     the launch read 13.6 GB past the L2s on the 600x248x248 front at 100
//     isovalues, tiled 7.4 GB; those reads reach 7 TB/s, also where the 256 MB
//     cache holds them).
//
// 600x248x248 front, 100 isovalues, 256 bins (5,050 pairs of 576,600 voxels):
// 3.04 -> 2.0 ms + 0.09 ms for the chains.  The counting's floor is its vector
// instructions, 11 per pair of values at 4 cycles per wave: 0.9 ms; on top come
// the rare exact divisions, LDS conflicts between lanes that meet in a counter
// (2.4e8 cycles over the CUs), the pairs' starts and the lists (0.3 ms), which
// one workgroup per CU cannot hide.  128 bins (2,080 pairs of 2^20 voxels, two
// workgroups per CU): 1.55 -> 1.12 ms (in 4 x 8 tiles alone 1.35); 256 bins,
// 2,016 pairs of 128^3 fields: 5.6 -> 3.4 ms; 256 isovalues of 60,000 voxels
// (32,896 pairs): 4.9 -> 2.1 ms.
#include "iso_internal.hpp"
#include "iso_bins.hpp"
#include "iso_nmi.hpp"

#include <algorithm>
#include <cfloat>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

namespace {

constexpr int kBlock = iso::kHistBlock;
constexpr int kWaves = kBlock / 64;
// Pairs of half a tile of the pair matrix (4 x 8), which is also the workgroups
// of 16-bit counters that an XCD runs at once (one per CU, 32 CUs).
constexpr int kTileRows = 4, kTileCols = 8, kTilePairs = kTileRows * kTileCols;
constexpr int kMaxTasksPerLaunch = 16384;  // one launch per 128-isovalue ISM (no tail wave)
constexpr size_t kMaxPartBytes = (size_t)128 << 20;  // slices' histograms of a launch

struct HistArgs {
  const float *fields;
  int64_t F;          // field size (N in the entropy normalisation)
  int64_t processed;  // voxels visited per pair (F, or fewer under Q16)
  const int2 *tasks;
  int ntasks;
  int slices;
  int64_t chunk;      // voxels per slice
  const float *mins;
  const float *maxs;
  uint32_t *ghist;    // ntasks * H*H, zero at rest
  uint32_t *arrive;   // ntasks, zero at rest
  uint32_t *parts;    // ntasks * slices LDS histograms, or null
  float *map;
  int n;
  int multi;
  int H;
  uint32_t *joint;
  uint32_t *rows;
  uint32_t *cols;
  int nxcd;
  int nmi32;     // reference float-order NMI (ISO_COMPAT_NMI32)
  int hist_bytes;         // LDS histogram
  iso::ChainBufs chains;  // nmi32: the chains' inputs, per task
};

// A wave-uniform value in a scalar register, however it was computed (integer
// divisions run on the vector unit): the fields' pointers that come from it then
// stay scalar, and their buffer loads need no per-lane waterfall.
__device__ __forceinline__ int scalar(int v) {
  asm volatile("" : "+v"(v));
  return __builtin_amdgcn_readfirstlane(v);
}

// Everything a workgroup keeps in LDS, the histogram first: at address 0 its
// atomics need no base added.
template <bool PACK16>
struct HistLds {
  iso::PairLds<PACK16> pair;
  double red[3][kWaves];
  uint32_t prog[2];
  int flushed, last;
};

// The pair's merged counts back into LDS, unless one needs more than its
// counter; returns where they are then (null: in LDS, and gh is zero again).
template <bool PACK16>
__device__ __forceinline__ uint32_t *take_back(uint32_t *s_hist, uint32_t *gh, int H) {
  const int tid = threadIdx.x, words = H * iso::kRowWords<PACK16>;
  bool fits = true;
  // several words per lane under way at a time: they come from beyond the L2
  constexpr int kAhead = 8;
  for (int w0 = tid; w0 < words; w0 += kAhead * kBlock) {
    uint32_t lo[kAhead], hi[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      const int w = w0 + q * kBlock;
      constexpr int kRow = iso::kRowWords<PACK16>;
      const int r = w / kRow, c = (PACK16 ? 2 : 1) * (w % kRow);
      lo[q] = w < words && c < H ? gh[r * H + c] : 0u;
      hi[q] = PACK16 && w < words && c + 1 < H ? gh[r * H + c + 1] : 0u;
    }
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      if (PACK16) fits &= (lo[q] | hi[q]) <= 0xffffu;
      if (w0 + q * kBlock < words) s_hist[w0 + q * kBlock] = lo[q] | hi[q] << 16;
    }
  }
  if (PACK16) fits = __syncthreads_and(fits);
  else __syncthreads();
  if (!fits) return gh;
  for (int e = tid; e < H * H; e += kBlock) gh[e] = 0u;  // zero at rest
  return nullptr;
}

// What comes of a pair's counts (in LDS, or in src): the joint histogram, the
// marginals, the NMI or the inputs of its chains.
template <bool PACK16>
__device__ __forceinline__ void finish_pair(const HistArgs &a, HistLds<PACK16> &s, uint32_t *s_hist,
                                            uint32_t *src, int task, int fi, int fj) {
  const int tid = threadIdx.x, H = a.H, HH = H * H;
  const bool mirror = !a.multi && fi != fj;
  const int mj = a.multi ? fj - a.n : fj;
  if (a.joint) {
    // the joint histogram out (and its transpose for the mirrored entry),
    // before the NMI reuses the LDS
    uint32_t *jout = a.joint + ((int64_t)fi * a.n + mj) * HH;
    uint32_t *jtr = mirror ? a.joint + ((int64_t)fj * a.n + fi) * HH : nullptr;
    for (int e = tid; e < HH; e += kBlock) {
      const uint32_t c = iso::pair_count<PACK16>(s_hist, src, H, e / H, e % H);
      jout[e] = c;
      if (jtr) jtr[(e % H) * H + e / H] = c;
    }
  }
  if (a.nmi32) {
    // ---- the chains of the reference's float order, folded by fold_kernel
    if (PACK16 && src)
      iso::emit_chains<PACK16, PACK16>(s_hist, a.hist_bytes, src, H, mirror, s.pair, a.chains, task);
    else
      iso::emit_chains<PACK16, false>(s_hist, a.hist_bytes, nullptr, H, mirror, s.pair, a.chains,
                                      task);
  } else {
    // ---- fused NMI from exact counts ----
    const double v = iso::nmi64_pair<PACK16>(s_hist, src, H, a.F, s.pair, s.red);
    if (tid == 0) {
      const float out = (v != v) ? 0.0f : (float)v;
      a.map[(int64_t)fi * a.n + mj] = out;
      if (mirror) a.map[(int64_t)fj * a.n + fi] = out;
    }
  }
  if (tid < H && a.rows) {  // (every form of the NMI ends its sums with a barrier)
    const uint32_t r = s.pair.rows[tid], c = s.pair.cols[tid];
    const int64_t o = ((int64_t)fi * a.n + mj) * H + tid;
    a.rows[o] = r;
    a.cols[o] = c;
    if (mirror) {
      const int64_t o2 = ((int64_t)fj * a.n + fi) * H + tid;
      a.rows[o2] = c;
      a.cols[o2] = r;
    }
  }
}

// STEP (picked by the autotuner): rounds of 8 values per lane and field on their
// way (16-bit counters), values per step (32-bit ones).
template <bool PACK16, int STEP>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(PACK16 ? 4 : 8))) void hist_nmi_kernel(HistArgs a) {
  extern __shared__ uint4 s_dyn[];
  uint32_t *s_hist = reinterpret_cast<uint32_t *>(s_dyn);
  HistLds<PACK16> &s = *reinterpret_cast<HistLds<PACK16> *>(s_hist + a.H * iso::kRowWords<PACK16>);

  const int tid = threadIdx.x;
  const int H = a.H;
  const int HH = H * H;
  const int words = H * iso::kRowWords<PACK16>;

  // Workgroups that run on an XCD at the same time take the pairs of one tile
  // of the pair matrix, slice by slice, so each value read serves several of
  // them from the XCD's L2.
  const uint32_t L = iso_xcd_remap(blockIdx.x, gridDim.x, (uint32_t)a.nxcd);
  const uint32_t per = (uint32_t)(kTilePairs * a.slices), tile = L / per, rem = L - tile * per;
  const uint32_t pairs = min((uint32_t)kTilePairs, (uint32_t)a.ntasks - tile * kTilePairs);
  const int task = scalar((int)(tile * kTilePairs + rem % pairs)), slice = scalar((int)(rem / pairs));
  const int2 tk = a.tasks[task];
  const int fi = tk.x, fj = tk.y;

  iso::clear_hist(s_hist, words);
  iso::clear_pair_lds(s.pair);
  if (tid == 0) { s.prog[0] = s.prog[1] = 0u; s.flushed = 0; s.last = 0; }

  iso::PairBins<PACK16> bin;
  {
    float mi = a.mins[fi], mj = a.mins[fj];
    float xi = a.maxs[fi], xj = a.maxs[fj];
    bin.init(mi < mj ? mi : mj, xi > xj ? xi : xj, H);
  }
  const int64_t begin = (int64_t)slice * a.chunk;
  const int len = (int)max((int64_t)0, min(a.chunk, a.processed - begin));
  const float *f1 = a.fields + (int64_t)fi * a.F + begin;
  const float *f2 = a.fields + (int64_t)fj * a.F + begin;
  uint32_t *gh = a.ghist + (int64_t)task * HH;
  __syncthreads();

  auto accumulate = [&](auto sub) {
    constexpr bool SUB = decltype(sub)::value;
    if constexpr (PACK16)
      iso::accumulate16<SUB, STEP>(bin, f1, f2, len, s_hist, s.prog, [&](int i, int j) {
        if (i >= H || j >= H) return;  // a value past the interval given
        atomicAdd(&gh[i * H + j], 32768u);
        s.flushed = 1;
      });
    else
      iso::accumulate32<SUB, STEP>(bin, f1, f2, len, s_hist);
  };
  if (__builtin_amdgcn_readfirstlane(bin.subtract)) accumulate(std::true_type());
  else accumulate(std::false_type());
  __syncthreads();

  if (a.parts && a.slices > 1) {
    // Slices of a pair meet in kernels of their own (merge_kernel,
    // finish_kernel), at whose start what was stored here is visible.  Added to
    // the pair's 32-bit histogram instead, with fences and a last workgroup that
    // takes the sum back, which is left for callers without room for the parts,
    // 136 pairs of 64^3 fields (128 bins, 3 slices) took 204 us with their
    // chains, now 108; 256 pairs of 2^20 voxels 307, now 182; 3 pairs of 4M
    // (256 bins, 85 slices) 165, now 141.  Stored here and added up by the last
    // workgroup, the release fences wrote the L2 back each time: 254 and 376 us.
    uint4 *const part = (uint4 *)(a.parts + ((int64_t)task * a.slices + slice) * words);
    for (int q = tid; q < words / 4; q += kBlock) part[q] = ((const uint4 *)s_hist)[q];
    return;
  }
  uint32_t *src = nullptr;  // where the pair's counts are, if not in LDS
  if (a.slices > 1 || s.flushed) {
    // LDS -> global 32-bit histogram of this task (columns past H hold counts
    // only for values past the interval given)
    for (int w = tid; w < words; w += kBlock) {
      const uint32_t v = s_hist[w];
      if (v) {
        const int r = w / iso::kRowWords<PACK16>, c = w % iso::kRowWords<PACK16>;
        if (PACK16) {
          const uint32_t lo = v & 0xffffu, hi = v >> 16;
          if (lo && 2 * c < H) atomicAdd(&gh[r * H + 2 * c], lo);
          if (hi && 2 * c + 1 < H) atomicAdd(&gh[r * H + 2 * c + 1], hi);
        } else if (c < H) {
          atomicAdd(&gh[r * H + c], v);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (a.slices > 1) {
      if (tid == 0) {
        uint32_t old = __hip_atomic_fetch_add(&a.arrive[task], 1u, __ATOMIC_ACQ_REL,
                                              __HIP_MEMORY_SCOPE_AGENT);
        s.last = (old == (uint32_t)a.slices - 1);
      }
      __syncthreads();
      if (!s.last) return;
    }
    // take_back reads with plain loads: no line of this CU's cache may be older
    // than the atomics (an odd H's histogram shares lines with the pair before)
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    src = take_back<PACK16>(s_hist, gh, H);
  }
  finish_pair<PACK16>(a, s, s_hist, src, task, fi, fj);
  if (tid == 0 && a.slices > 1) a.arrive[task] = 0u;
}

// The slices' histograms of a pair, added up into its 32-bit one (which holds
// what 16-bit counters handed on).  A lane per 16 bytes of a histogram.
template <bool PACK16>
__global__ __launch_bounds__(256) void merge_kernel(HistArgs a) {
  const int quads = a.H * iso::kRowWords<PACK16> / 4, q = blockIdx.x * 256 + threadIdx.x;
  if (q >= quads) return;
  const uint4 *part = (const uint4 *)a.parts + (int64_t)blockIdx.y * a.slices * quads + q;
  uint32_t lo[4] = {}, hi[4] = {};
#pragma unroll 8
  for (int k = 0; k < a.slices; ++k) {
    const uint4 v = part[(int64_t)k * quads];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] += PACK16 ? w[e] & 0xffffu : w[e];
      if (PACK16) hi[e] += w[e] >> 16;
    }
  }
  constexpr int kRow = iso::kRowWords<PACK16>;
  const int H = a.H, row = 4 * q / kRow, w = 4 * q % kRow;
  uint32_t *gh = a.ghist + (int64_t)blockIdx.y * H * H + row * H;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = (PACK16 ? 2 : 1) * (w + e);
    if (lo[e] && c < H) gh[c] += lo[e];
    if (PACK16 && hi[e] && c + 1 < H) gh[c + 1] += hi[e];
  }
}

// ... and what comes of the merged counts, a workgroup per pair.
template <bool PACK16>
__global__ __launch_bounds__(kBlock) void finish_kernel(HistArgs a) {
  extern __shared__ uint4 s_dyn[];
  uint32_t *s_hist = reinterpret_cast<uint32_t *>(s_dyn);
  HistLds<PACK16> &s = *reinterpret_cast<HistLds<PACK16> *>(s_hist + a.H * iso::kRowWords<PACK16>);
  const int task = blockIdx.x;
  const int2 tk = a.tasks[task];
  iso::clear_pair_lds(s.pair);
  uint32_t *src = take_back<PACK16>(s_hist, a.ghist + (int64_t)task * a.H * a.H, a.H);
  finish_pair<PACK16>(a, s, s_hist, src, task, tk.x, tk.y);
}

// The float-order NMI of every task of a hist_nmi_kernel launch: kFoldPairs
// tasks per workgroup.
__global__ __launch_bounds__(64 * iso::kFoldWaves) void fold_kernel(HistArgs a) {
  __shared__ iso::FoldLds s_fold;
  const int64_t t0 = (int64_t)blockIdx.x * iso::kFoldPairs;
  iso::fold_chains(a.chains, a.H, t0, a.ntasks, [&](int64_t t) {
    const int2 tk = a.tasks[t];
    const int mj = a.multi ? tk.y - a.n : tk.y;
    return iso::FoldOut{!a.multi && tk.x != tk.y, a.F, a.map + (int64_t)tk.x * a.n + mj,
                        a.map + (int64_t)tk.y * a.n + tk.x};
  }, s_fold);
}

// logf of the counts 1 to kLogs - 1, 0 for 0
__global__ void logs_kernel(float *logs) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < iso::kLogs) logs[c] = c ? iso::logf_cr((float)c) : 0.0f;
}

// ---- per-field (min, max), DistanceField::getInterval semantics ----
constexpr int kIntBlock = 256;

__global__ __launch_bounds__(kIntBlock) void interval_partial_kernel(const float *fields, int64_t F,
                                                                     int parts, float2 *part) {
  const int field = blockIdx.y;
  const int p = blockIdx.x;
  const float *f = fields + (int64_t)field * F;
  int64_t chunk = (F + parts - 1) / parts;
  int64_t b = (int64_t)p * chunk, e = b + chunk;
  if (e > F) e = F;
  // min and max by these comparisons ignore NaN and, over values that are
  // never -0 (distances), do not depend on the order they are taken in
  float lo = FLT_MAX, hi = FLT_MIN;
  int64_t i = b + threadIdx.x;
  for (; i + 3 * kIntBlock < e; i += 4 * kIntBlock) {  // four loads in flight
    const float v[4] = {f[i], f[i + kIntBlock], f[i + 2 * kIntBlock], f[i + 3 * kIntBlock]};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      lo = v[u] < lo ? v[u] : lo;
      hi = v[u] > hi ? v[u] : hi;
    }
  }
  for (; i < e; i += kIntBlock) {
    const float v = f[i];
    lo = v < lo ? v : lo;
    hi = v > hi ? v : hi;
  }
  __shared__ float s_lo[kIntBlock / 64], s_hi[kIntBlock / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float l2 = __shfl_xor(lo, o, 64), h2 = __shfl_xor(hi, o, 64);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  if ((threadIdx.x & 63) == 0) { s_lo[threadIdx.x >> 6] = lo; s_hi[threadIdx.x >> 6] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kIntBlock / 64; ++k) {
      lo = s_lo[k] < lo ? s_lo[k] : lo;
      hi = s_hi[k] > hi ? s_hi[k] : hi;
    }
    part[(int64_t)field * parts + p] = make_float2(lo, hi);
  }
}

__global__ void interval_final_kernel(const float2 *part, int parts, int nfields, float *mins,
                                      float *maxs) {
  int field = blockIdx.x * blockDim.x + threadIdx.x;
  if (field >= nfields) return;
  float lo = FLT_MAX, hi = FLT_MIN;
  for (int p = 0; p < parts; ++p) {
    float2 v = part[(int64_t)field * parts + p];
    lo = v.x < lo ? v.x : lo;
    hi = v.y > hi ? v.y : hi;
  }
  mins[field] = lo;
  maxs[field] = hi;
}

}  // namespace

namespace iso {

int field_interval(iso_ctx *ctx, const float *d_fields, int nfields, int64_t F, float *d_mins,
                   float *d_maxs) {
  // about 16K values per workgroup: enough workgroups to fill the chip
  int parts = (int)std::min<int64_t>(256, (F + 16383) / 16384);
  if (parts < 1) parts = 1;
  void *part = nullptr;
  ISO_TRY(ws_get(ctx, WS_INTERVAL_PART, sizeof(float2) * (size_t)parts * nfields, false, &part));
  hipLaunchKernelGGL(interval_partial_kernel, dim3(parts, nfields), dim3(kIntBlock), 0,
                     ctx->stream, d_fields, F, parts, (float2 *)part);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  hipLaunchKernelGGL(interval_final_kernel, dim3((nfields + 127) / 128), dim3(128), 0, ctx->stream,
                     (const float2 *)part, parts, nfields, d_mins, d_maxs);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

int nmi_logs_fill(iso_ctx *ctx, float *d_logs) {
  hipLaunchKernelGGL(logs_kernel, dim3(kLogs / 256), dim3(256), 0, ctx->stream, d_logs);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

int nmi_logs(iso_ctx *ctx, const float **out) {
  const bool first = !ctx->ws[WS_NMI_LOGS].ptr;
  void *p = nullptr;
  ISO_TRY(ws_get(ctx, WS_NMI_LOGS, sizeof(float) * kLogs, false, &p));
  if (first) ISO_TRY(nmi_logs_fill(ctx, (float *)p));
  *out = (const float *)p;
  return ISO_OK;
}

int chain_tasks(const iso_ctx *ctx, int H, int64_t F, int64_t ntasks, int limit_mib) {
  size_t limit = (size_t)limit_mib << 20;
  if (const char *e = std::getenv("ISO_NMI_CHAIN_MIB")) {  // read per call
    const long v = std::atol(e);
    if (v > 0) limit = (size_t)std::min<long>(v, 65536) << 20;
  }
  // (a workspace that grows takes a quarter more)
  const int64_t fit = (int64_t)(limit / 5 * 4 / chain_task_bytes(H, F));
  const int64_t round = (int64_t)(H > 128 ? 1 : 2) * ctx->cu_count;
  const int64_t most = fit >= round ? fit / round * round : std::max<int64_t>(1, fit);
  return (int)std::min<int64_t>(most, std::min<int64_t>(ntasks, INT32_MAX));
}

int chain_get(iso_ctx *ctx, int64_t ntasks, int H, int64_t F, ChainBufs &b) {
  void *p = nullptr;
  ISO_TRY(ws_get(ctx, WS_NMI_CHAINS, chain_task_bytes(H, F) * (size_t)ntasks + kChainPad, false, &p));
  chain_carve(b, p, ntasks, H, F);
  return nmi_logs(ctx, &b.logs);
}

// Slices per pair, where the pairs alone leave CUs idle (one workgroup per CU
// with 16-bit counters, two with 32-bit ones): as few rounds of voxels as
// possible, a slice counting another 32K voxels' time for its start and the
// merge (10 us at 3 voxels per ns), with at least 16K voxels each (16 pairs of
// 262,144, 128 bins, by another 32K, 16K, 8K: 108, 109, 122 us).
// With a round or more of pairs, slices would only add merges (2,016 pairs of
// 128^3 fields, 256 bins: 3.7 ms, cut up to even the last round out 7.0 ms).
static int64_t slice_count(const iso_ctx *ctx, int64_t processed, int64_t nt, bool pack16) {
  const int64_t cap = (int64_t)(pack16 ? 1 : 2) * ctx->cu_count;
  int64_t slices = 1, best = INT64_MAX;
  for (int64_t k = 1; nt < cap && k <= std::max<int64_t>(1, processed / 16384); ++k) {
    const int64_t rounds = (nt * k + cap - 1) / cap;
    // (no larger k can cost less than its rounds' starts and the voxels' share)
    if (rounds * 32768 + nt * (processed - k) / cap > best) break;
    const int64_t cost = rounds * (processed / k + (k > 1 ? 32768 : 0));
    if (cost < best) {
      best = cost;
      slices = k;
    }
  }
  return std::max(slices, (processed + kMaxSlice - 1) / kMaxSlice);
}

static int64_t processed_voxels(int64_t F, uint32_t flags) {
  const int64_t C = 1000000;
  return (flags & ISO_COMPAT_HIST_CHUNKS) && F > 0 && F % C == 0 ? F - C : F;
}

size_t hist_parts_bytes(const iso_ctx *ctx, int64_t F, int H, uint32_t flags, int64_t nt) {
  const int64_t slices = slice_count(ctx, processed_voxels(F, flags), nt, H > 128);
  return slices > 1 ? sizeof(uint32_t) * (size_t)(nt * slices) * H * row_words(H) : 0;
}

// Launches the histogram+NMI kernel over a device task list.
int hist_nmi_tasks(iso_ctx *ctx, const float *d_fields, int n, int64_t F, int H, int multi,
                   uint32_t flags, const float *d_mins, const float *d_maxs, float *d_map,
                   const int2 *d_tasks, int ntasks, uint32_t *d_joint, uint32_t *d_rows,
                   uint32_t *d_cols) {
  if (ntasks <= 0) return ISO_OK;
  const bool pack16 = H > 128;
  const bool nmi32 = (flags & ISO_COMPAT_NMI32) != 0;
  HistBufs b;
  int most = kMaxTasksPerLaunch;
  if (nmi32) {
    most = std::min(most, chain_tasks(ctx, H, F, ntasks, pack16 ? 2048 : 1024));
    ISO_TRY(chain_get(ctx, most, H, F, b.chains));
  }
  const int64_t processed = processed_voxels(F, flags);
  auto run = [&](int variant) -> int {
    for (int t0 = 0; t0 < ntasks; t0 += most) {
      const int nt = std::min(ntasks - t0, most);
      void *gh = nullptr, *arr = nullptr;
      ISO_TRY(ws_get(ctx, WS_HIST_GLOBAL, sizeof(uint32_t) * (size_t)nt * H * H, true, &gh));
      ISO_TRY(ws_get(ctx, WS_HIST_ARRIVE, sizeof(uint32_t) * (size_t)nt, true, &arr));
      b.ghist = (uint32_t *)gh;
      b.arrive = (uint32_t *)arr;
      // the slices' histograms: a few hundred workgroups' (only a slice past
      // kMaxSlice voxels comes with more pairs than that)
      const size_t pb = hist_parts_bytes(ctx, F, H, flags, nt);
      void *parts = nullptr;
      if (pb > 0 && pb <= kMaxPartBytes)
        ISO_TRY(ws_get(ctx, WS_HIST_PARTS, pb, false, &parts));
      b.parts = (uint32_t *)parts;
      ISO_TRY(hist_launch(ctx, d_fields, n, F, H, multi, flags, d_mins, d_maxs, d_map,
                          d_tasks + t0, nt, d_joint, d_rows, d_cols, b, variant));
    }
    return ISO_OK;
  };
  const uint64_t key = ((uint64_t)H << 32) | ((uint64_t)ceil_log2((uint64_t)processed) << 16) |
                       (uint64_t)ceil_log2((uint64_t)ntasks);
  return tune_pick(ctx, kTuneHist, key, {0, 1}, 1,
                   pack16 ? "hist16 rounds ahead {0: 1, 1: 2}" : "hist32 loads/step {0: 4, 1: 8}", run);
}

// One launch of the histogram + NMI kernels over nt tasks with the caller's
// buffers (ghist: nt * H * H words and arrive: nt words, both zero at rest;
// for ISO_COMPAT_NMI32 the chains' inputs of nt tasks and the logarithms).
// Launch variant 0 or 1 (the autotuner's choices).
int hist_launch(iso_ctx *ctx, const float *d_fields, int n, int64_t F, int H, int multi,
                uint32_t flags, const float *d_mins, const float *d_maxs, float *d_map,
                const int2 *d_tasks, int nt, uint32_t *d_joint, uint32_t *d_rows,
                uint32_t *d_cols, const HistBufs &b, int variant) {
  if (nt <= 0) return ISO_OK;
  const bool pack16 = H > 128;
  const bool nmi32 = (flags & ISO_COMPAT_NMI32) != 0;
  const size_t hist_bytes = sizeof(uint32_t) * (size_t)H * row_words(H);
  const size_t lds = hist_bytes + (pack16 ? sizeof(HistLds<true>) : sizeof(HistLds<false>));
  const int64_t processed = processed_voxels(F, flags);
  // variants: 16-bit counters with 1 or 2 rounds of 8 values on their way,
  // 32-bit counters with 4 or 8 values per step (the autotuner picks; 16 would
  // take too many registers for two workgroups per CU).  The LDS limit is
  // raised once per process, whatever thread gets here.
  static std::once_flag attr_once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(attr_once, [] {
    const void *kern[6] = {(const void *)hist_nmi_kernel<false, 4>,
                           (const void *)hist_nmi_kernel<false, 8>,
                           (const void *)hist_nmi_kernel<true, 1>,
                           (const void *)hist_nmi_kernel<true, 2>,
                           (const void *)finish_kernel<false>,
                           (const void *)finish_kernel<true>};
    for (int v = 0; v < 6 && attr_err == hipSuccess; ++v)
      attr_err = hipFuncSetAttribute(
          kern[v], hipFuncAttributeMaxDynamicSharedMemorySize,
          v < 2 || v == 4 ? 128 * 4 * kRowWords<false> + (int)sizeof(HistLds<false>)
                          : 256 * 4 * kRowWords<true> + (int)sizeof(HistLds<true>));
  });
  ISO_HIP_CHECK(ctx, attr_err);
  const int64_t slices = slice_count(ctx, processed, nt, pack16);
  const int64_t chunk = (processed + slices - 1) / slices;
  HistArgs a;
  a.fields = d_fields;
  a.F = F;
  a.processed = processed;
  a.tasks = d_tasks;
  a.ntasks = nt;
  a.slices = (int)slices;
  a.chunk = chunk;
  a.mins = d_mins;
  a.maxs = d_maxs;
  a.ghist = b.ghist;
  a.arrive = b.arrive;
  a.parts = b.parts;
  a.map = d_map;
  a.n = n;
  a.multi = multi;
  a.H = H;
  a.joint = d_joint;
  a.rows = d_rows;
  a.cols = d_cols;
  a.nxcd = ctx->xcd_count;
  a.nmi32 = nmi32 ? 1 : 0;
  a.hist_bytes = (int)hist_bytes;
  a.chains = b.chains;
  dim3 grid((unsigned)(nt * slices));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, ctx->stream, a);
  };
  if (pack16) variant == 0 ? launch(hist_nmi_kernel<true, 1>) : launch(hist_nmi_kernel<true, 2>);
  else variant == 0 ? launch(hist_nmi_kernel<false, 4>) : launch(hist_nmi_kernel<false, 8>);
  if (a.parts && slices > 1) {
    const dim3 mg((unsigned)((H * row_words(H) / 4 + 255) / 256), (unsigned)nt);
    if (pack16) {
      hipLaunchKernelGGL(merge_kernel<true>, mg, dim3(256), 0, ctx->stream, a);
      hipLaunchKernelGGL(finish_kernel<true>, dim3((unsigned)nt), dim3(kBlock), lds, ctx->stream, a);
    } else {
      hipLaunchKernelGGL(merge_kernel<false>, mg, dim3(256), 0, ctx->stream, a);
      hipLaunchKernelGGL(finish_kernel<false>, dim3((unsigned)nt), dim3(kBlock), lds, ctx->stream, a);
    }
  }
  ISO_HIP_CHECK(ctx, hipGetLastError());
  if (nmi32)
    hipLaunchKernelGGL(fold_kernel, dim3((unsigned)((nt + kFoldPairs - 1) / kFoldPairs)),
                       dim3(64 * kFoldWaves), 0, ctx->stream, a);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  return ISO_OK;
}

// Unordered pairs (i <= j), or all n*n pairs (i, n + j) for multi, in tiles of 8
// x 8, the upper four rows first.
void build_tasks(int n, int multi, std::vector<int2> &t) {
  t.clear();
  for (int i0 = 0; i0 < n; i0 += 2 * kTileRows)
    for (int j0 = multi ? 0 : i0; j0 < n; j0 += kTileCols)
      for (int h = i0; h < std::min(i0 + 2 * kTileRows, n); h += kTileRows)
        for (int i = h; i < std::min(h + kTileRows, n); ++i)
          for (int j = multi ? j0 : std::max(i, j0); j < std::min(j0 + kTileCols, n); ++j)
            t.push_back(make_int2(i, multi ? n + j : j));
}

}  // namespace iso

extern "C" {

int iso_field_interval(iso_ctx *ctx, const float *d_fields, int nfields, int64_t F,
                       float *d_mins, float *d_maxs) {
  ISO_TRY(iso::enter(ctx));
  if (!d_fields || !d_mins || !d_maxs || nfields <= 0 || F <= 0)
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_field_interval: bad arguments");
  return iso::field_interval(ctx, d_fields, nfields, F, d_mins, d_maxs);
}

int iso_hist_nmi(iso_ctx *ctx, const float *d_fields, int n, int64_t F, int H, int multi,
                 uint32_t flags, const float *d_mins, const float *d_maxs, float *d_map,
                 uint32_t *d_joint, uint32_t *d_rows, uint32_t *d_cols) {
  ISO_TRY(iso::enter(ctx));
  if (!d_fields || !d_mins || !d_maxs || !d_map || n <= 0 || F <= 0)
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_hist_nmi: bad arguments");
  if (H < 1 || H > 256)
    return iso::fail(ctx, ISO_ERR_UNSUPPORTED, "iso_hist_nmi: H=%d outside [1,256]", H);
  if ((d_rows == nullptr) != (d_cols == nullptr))
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_hist_nmi: rows and cols go together");
  std::vector<int2> tasks;
  iso::build_tasks(n, multi, tasks);
  void *dt = nullptr, *pin = nullptr;
  size_t tb = sizeof(int2) * tasks.size();
  ISO_TRY(iso::ws_get(ctx, WS_HIST_TASKS, tb, false, &dt));
  ISO_TRY(iso::pinned_get(ctx, tb, &pin));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));  // pinned buffer reuse
  memcpy(pin, tasks.data(), tb);
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(dt, pin, tb, hipMemcpyHostToDevice, ctx->stream));
  ISO_TRY(iso::hist_nmi_tasks(ctx, d_fields, n, F, H, multi, flags, d_mins, d_maxs, d_map,
                              (const int2 *)dt, (int)tasks.size(), d_joint, d_rows, d_cols));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return ISO_OK;
}

}  // extern "C"
