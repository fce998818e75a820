// Volume ingest and isovalue selection, the front of the `single` module.
//
// Ingest (filehandler/src/BinaryFloatReader.cpp:29-49, types/src/Isosurface.cpp:
// 32-76, 185-200): a raw float32 file stored x-fastest becomes the z-fastest
// image img[(x*Y + y)*Z + z] = file[x + y*X + z*X*Y]; realMin/realMax are the
// extremes of the values inside [cfg.min, cfg.max], starting from 100000 and
// -100000.  Here: an LDS-tiled 64x64 transpose per y plane (reads coalesced
// along x, writes along z) with the restricted min/max folded in.
//
// Isovalues (runtime/src/Single.cpp:286-392, uniform = true): a 65536-bin
// histogram of the image over [realMin, realMax] on the device, then the
// reference's equalisation walk over the bins on the host (128 bins at a step).
// Bin index = int(65536 * (v - gmin) * oneovergrange) with oneovergrange the
// float of 1.0/(double)(gmax - gmin), clamped to [0, 65535]; the reference's
// loop bound is a float (dataSize), so voxel i counts iff float(i) < float(n).
#include <algorithm>
#include <cstring>

#include "iso_internal.hpp"

namespace {

constexpr int kT = 64;

// Transposes 64 x 64 tiles (x by z at one y), the loads of a workgroup's next
// tile in flight while it writes the current one.  Bound by memory: every
// voxel is read and written once, and the 256-byte rows on both sides keep
// partly used lines rare where X or Z is not a multiple of 32; the tiles run
// along the file's rows.  600x248x248: 109 -> 75 us (3.9 TB/s; a plain copy
// reaches 4.7).
__global__ __launch_bounds__(256) void ingest_kernel(const float *file, int X, int Y, int Z,
                                                     int tx_n, int tz_n, int64_t tiles, float cmin,
                                                     float cmax, float *img, float2 *part) {
  __shared__ float tile[kT][kT + 1];
  __shared__ float s_lo[4], s_hi[4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  float lo = 100000.0f, hi = -100000.0f;
  float v[kT / 4];
  int x0, y, z0;
  auto place = [&](int64_t t) {
    x0 = (int)(t % tx_n) * kT;
    y = (int)(t / tx_n % Y);
    z0 = (int)(t / tx_n / Y) * kT;
  };
  auto load = [&]() {
    const int x = x0 + lane;
    const float *src = file + x + (int64_t)y * X;
#pragma unroll
    for (int r = 0; r < kT / 4; ++r) {
      const int z = z0 + w + 4 * r;
      if (x < X && z < Z) v[r] = src[(int64_t)z * X * Y];
    }
  };
  int64_t t = blockIdx.x;
  place(t);
  load();
  while (true) {
    const int x1 = x0, y1 = y, z1 = z0;
#pragma unroll
    for (int r = 0; r < kT / 4; ++r) {
      if (x1 + lane < X && z1 + w + 4 * r < Z) {
        tile[w + 4 * r][lane] = v[r];
        if (v[r] < lo && v[r] >= cmin) lo = v[r];
        if (v[r] > hi && v[r] <= cmax) hi = v[r];
      }
    }
    __syncthreads();
    t += gridDim.x;
    if (t < tiles) {
      place(t);
      load();
    }
    if (z1 + lane < Z) {
#pragma unroll
      for (int r = 0; r < kT / 4; ++r) {
        const int x = x1 + w + 4 * r;
        if (x < X) img[((int64_t)x * Y + y1) * Z + z1 + lane] = tile[lane][w + 4 * r];
      }
    }
    if (t >= tiles) break;
    __syncthreads();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float l2 = __shfl_xor(lo, o, 64), h2 = __shfl_xor(hi, o, 64);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  if (lane == 0) { s_lo[w] = lo; s_hi[w] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 4; ++i) {
      lo = s_lo[i] < lo ? s_lo[i] : lo;
      hi = s_hi[i] > hi ? s_hi[i] : hi;
    }
    part[blockIdx.x] = make_float2(lo, hi);
  }
}

__global__ void minmax_final_kernel(const float2 *part, int64_t n, float2 *out) {
  __shared__ float s_lo[16], s_hi[16];
  float lo = 100000.0f, hi = -100000.0f;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    float2 v = part[i];
    lo = v.x < lo ? v.x : lo;
    hi = v.y > hi ? v.y : hi;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float l2 = __shfl_xor(lo, o, 64), h2 = __shfl_xor(hi, o, 64);
    lo = l2 < lo ? l2 : lo;
    hi = h2 > hi ? h2 : hi;
  }
  if ((threadIdx.x & 63) == 0) { s_lo[threadIdx.x >> 6] = lo; s_hi[threadIdx.x >> 6] = hi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
      lo = s_lo[w] < lo ? s_lo[w] : lo;
      hi = s_hi[w] > hi ? s_hi[w] : hi;
    }
    *out = make_float2(lo, hi);
  }
}

constexpr int kBins = 65536;
constexpr int kHistRound = 4096;  // voxels a workgroup takes at a time, four per lane
constexpr int kHistEpoch = 8;     // rounds between barriers
constexpr int kBlockBins = 128;   // bins of one block sum
constexpr int kBinBlocks = kBins / kBlockBins;

struct __attribute__((packed, aligned(4))) float4u {
  float v[4];
};

__device__ __forceinline__ uint32_t equal_bin(float v, float gmin, float oneover) {
  int idx = (int)(((float)kBins * (v - gmin)) * oneover);
  idx = idx > kBins - 1 ? kBins - 1 : idx;
  return (uint32_t)(idx < 0 ? 0 : idx);
}

// Each workgroup keeps all 65536 bins in its LDS as 16-bit counters, two per
// word (128 KB), and writes them out once; sum_hist_kernel adds them up.  The
// lane whose add carries a counter to 32,768 takes that much out again into
// the global `over`.  Between two barriers a counter gains at most kHistEpoch
// rounds, 32,768, and at a barrier it is below 32,768: it never reaches 2^16.
// Voxels are clustered (a plateau's all fall into one bin), so a wave first
// counts those that share its first lane's bin and adds them at once; only the
// others queue up in the LDS.  600x248x248 front: 50 us and 6 us for the sums,
// 2.9 TB/s against 7 that reading reaches; with one global atomic per voxel
// the front's plateaus took 109 ms.
__global__ __launch_bounds__(1024) void uniform_hist_kernel(const float *img, int64_t n, float gmin,
                                                            float oneover, uint32_t *over,
                                                            uint32_t *parts) {
  extern __shared__ uint32_t s_cnt[];  // kBins / 2
  for (int i = threadIdx.x; i < kBins / 8; i += 1024) ((uint4 *)s_cnt)[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  const int64_t rounds = (n + kHistRound - 1) / kHistRound;
  const int lane = threadIdx.x & 63;
  auto load = [&](int64_t r) {
    float4u f = {};
    const int64_t i = r * kHistRound + threadIdx.x * 4;
    if (i + 4 <= n)
      f = *(const float4u *)(img + i);
    else
      for (int j = 0; j < 3; ++j)
        if (i + j < n) f.v[j] = img[i + j];
    return f;
  };
  int64_t r = blockIdx.x;
  float4u nxt = load(r);
  for (int t = 0; r < rounds; ++t) {
    if (t == kHistEpoch) {
      __syncthreads();
      t = 0;
    }
    const float4u cur = nxt;
    const int64_t i0 = r * kHistRound + threadIdx.x * 4;
    r += gridDim.x;
    if (r < rounds) nxt = load(r);
    uint32_t b[4], amount[4], old[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      b[j] = equal_bin(cur.v[j], gmin, oneover);
      const bool in = i0 + j < n;
      const uint32_t first = __builtin_amdgcn_readfirstlane(b[j]);
      const uint64_t same = __ballot(in && b[j] == first);
      amount[j] = lane == 0 ? (uint32_t)__popcll(same) : (in && b[j] != first) ? 1u : 0u;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (amount[j]) old[j] = atomicAdd(&s_cnt[b[j] >> 1], amount[j] << (16 * (b[j] & 1)));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!amount[j]) continue;
      const uint32_t sh = 16 * (b[j] & 1), c = (old[j] >> sh) & 0xffff;
      if (c < 0x8000u && c + amount[j] >= 0x8000u) {
        atomicSub(&s_cnt[b[j] >> 1], 0x8000u << sh);
        atomicAdd(&over[b[j]], 0x8000u);
      }
    }
  }
  __syncthreads();
  uint4 *out = (uint4 *)(parts + (int64_t)blockIdx.x * (kBins / 2));
  for (int i = threadIdx.x; i < kBins / 8; i += 1024) out[i] = ((const uint4 *)s_cnt)[i];
}

// bins[] += the workgroups' counters, and the sums of each 128 bins.  One
// workgroup per block of bins: lane = word, the parts split over its waves.
__global__ __launch_bounds__(1024) void sum_hist_kernel(const uint32_t *parts, int nparts,
                                                        uint32_t *bins, int64_t *blocks) {
  __shared__ uint32_t s_lo[16][64], s_hi[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t *src = parts + (int64_t)blockIdx.x * 64 + lane;
  uint32_t lo = 0, hi = 0;
#pragma unroll 4
  for (int p = w; p < nparts; p += 16) {
    const uint32_t c = src[(int64_t)p * (kBins / 2)];
    lo += c & 0xffff;
    hi += c >> 16;
  }
  s_lo[w][lane] = lo;
  s_hi[w][lane] = hi;
  __syncthreads();
  if (w) return;
  for (int i = 1; i < 16; ++i) {
    lo += s_lo[i][lane];
    hi += s_hi[i][lane];
  }
  uint2 *at = (uint2 *)bins + blockIdx.x * 64 + lane;
  uint2 c = *at;
  c.x += lo;
  c.y += hi;
  *at = c;
  int64_t sum = (int64_t)(int)c.x + (int)c.y;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  if (lane == 0) blocks[blockIdx.x] = sum;
}

}  // namespace

extern "C" {

int iso_volume_ingest(iso_ctx *ctx, const float *d_file, int X, int Y, int Z, float cfg_min,
                      float cfg_max, float *d_img, float *h_real_min, float *h_real_max) {
  ISO_TRY(iso::enter(ctx));
  if (!d_file || !d_img || X <= 0 || Y <= 0 || Z <= 0 || d_file == d_img)
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_volume_ingest: bad arguments");
  const int tx_n = (X + kT - 1) / kT, tz_n = (Z + kT - 1) / kT;
  const int64_t tiles = (int64_t)tx_n * tz_n * Y;
  // as many workgroups as the LDS of the CUs holds
  const int64_t nb = std::min<int64_t>(tiles, 8 * (int64_t)ctx->cu_count);
  void *part = nullptr, *res = nullptr, *hb = nullptr;
  ISO_TRY(iso::ws_get(ctx, WS_INTERVAL_PART, sizeof(float2) * (size_t)nb, false, &part));
  ISO_TRY(iso::ws_get(ctx, WS_SMALL, 64, false, &res));
  ISO_TRY(iso::pinned_get(ctx, sizeof(float2), &hb));
  hipLaunchKernelGGL(ingest_kernel, dim3((unsigned)nb), dim3(256), 0, ctx->stream, d_file, X, Y, Z,
                     tx_n, tz_n, tiles, cfg_min, cfg_max, d_img, (float2 *)part);
  hipLaunchKernelGGL(minmax_final_kernel, dim3(1), dim3(1024), 0, ctx->stream,
                     (const float2 *)part, nb, (float2 *)res);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(hb, res, sizeof(float2), hipMemcpyDeviceToHost, ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  const float2 mm = *(const float2 *)hb;
  if (h_real_min) *h_real_min = mm.x;
  if (h_real_max) *h_real_max = mm.y;
  return ISO_OK;
}

int iso_equalized_isovalues(iso_ctx *ctx, const float *d_img, int64_t n, float real_min,
                            float real_max, int k, float *h_isos) {
  ISO_TRY(iso::enter(ctx));
  if (!d_img || n <= 0 || k <= 0 || !h_isos)
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_equalized_isovalues: bad arguments");
  // (of the context's device: a process may hold contexts on several)
  ISO_HIP_CHECK(ctx, hipFuncSetAttribute((const void *)uniform_hist_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, kBins * 2));
  // voxel i counts iff float(i) < float(n): those below the first that does not
  const float fn = (float)n;
  int64_t counted = 0;
  for (int64_t hi = n; counted < hi;) {
    const int64_t mid = counted + (hi - counted) / 2;
    if ((float)mid < fn)
      counted = mid + 1;
    else
      hi = mid;
  }
  // one workgroup per CU, each with at least an epoch of rounds: its counters
  // cost 128 KB to clear, write out and add up
  const int64_t epochs = (n + (int64_t)kHistRound * kHistEpoch - 1) / (kHistRound * kHistEpoch);
  const int groups = (int)std::min<int64_t>(epochs, ctx->cu_count);
  const size_t bin_bytes = sizeof(uint32_t) * kBins, sum_bytes = sizeof(int64_t) * kBinBlocks;
  void *dh = nullptr, *hb = nullptr;
  ISO_TRY(iso::ws_get(ctx, WS_MC_KEYS_B,
                      bin_bytes + sum_bytes + sizeof(uint32_t) * (kBins / 2) * (size_t)groups,
                      false, &dh));
  ISO_TRY(iso::pinned_get(ctx, bin_bytes + sum_bytes, &hb));
  uint32_t *parts = (uint32_t *)((char *)dh + bin_bytes + sum_bytes);
  ISO_TRY(iso::fill_u32(ctx, dh, 0u, kBins));
  const float oneover = (float)(1.0 / (double)(real_max - real_min));
  hipLaunchKernelGGL(uniform_hist_kernel, dim3((unsigned)groups), dim3(1024), kBins * 2,
                     ctx->stream, d_img, counted, real_min, oneover, (uint32_t *)dh, parts);
  hipLaunchKernelGGL(sum_hist_kernel, dim3(kBinBlocks), dim3(1024), 0, ctx->stream, parts, groups,
                     (uint32_t *)dh, (int64_t *)((char *)dh + bin_bytes));
  ISO_HIP_CHECK(ctx, hipGetLastError());
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(hb, dh, bin_bytes + sum_bytes, hipMemcpyDeviceToHost,
                                    ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  const int *hist = (const int *)hb;
  const int64_t *sums = (const int64_t *)((const char *)hb + bin_bytes);
  // Equalisation walk (Single.cpp:362-389): isovalue i takes bins until the next
  // would reach its share of what is left.  All sums are whole numbers, exact
  // in double, so 128 bins whose sum stays below the share are taken at once
  // (counts past 2^31 are negative as int: bin by bin, as the reference).
  const bool jump = n <= INT32_MAX;
  double sum = 0.0, acc = 0.0, threshold;
  for (int b = 0; b < kBinBlocks; ++b) sum += (double)sums[b];
  int index = 0;
  threshold = sum / double(k);
  for (int i = 0; i < k; ++i) {
    while (index < kBins - 1) {
      if (jump && index % kBlockBins == 0 && index < kBins - kBlockBins) {
        const double s = (double)sums[index / kBlockBins];
        if (acc == 0.0 ? s == 0.0 : acc + s < threshold) {
          acc += s;
          index += kBlockBins;
          continue;
        }
      }
      if (acc != 0.0 && !(acc + hist[index] < threshold)) break;
      acc += hist[index++];
    }
    std::memcpy(&h_isos[i], &index, sizeof index);  // until it becomes the isovalue
    sum -= acc;
    acc = 0.0;
    if (i < k - 1) threshold = sum / double(k - (i + 1));
  }
  // bins -> isovalues (Single.cpp:304-319)
  // The reference relabels a bin with its isovalue and passes bins up to i: those
  // of isovalues up to i, and past the last isovalue's the bins left with their
  // counts.
  int idx = 0, last = 0;
  const float step = (real_max - real_min) / (float)kBins;
  for (int i = 0; i < k; ++i) {
    int end;
    std::memcpy(&end, &h_isos[i], sizeof end);
    if (idx < end) idx = end;
    if (idx >= index)
      while (idx < kBins && hist[idx] <= i) ++idx;
    const int range = idx - last;
    const int mid = last + range / 2;
    const float off = step * (float)mid;
    h_isos[i] = real_min + off;
    last = idx;
  }
  return ISO_OK;
}

}  // extern "C"
