// Exact histogram binning shared by the histogram kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace iso {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// floor(v), 0 for a negative v or a NaN (what v_cvt_u32_f32 does; the
// language leaves those conversions undefined).
__device__ __forceinline__ uint32_t floor_u32(float v) {
  uint32_t r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// Both halves' unsigned maximum (v_pk_max_u16).
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(
      uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// a's high half times k, plus c.
__device__ __forceinline__ uint32_t mad_hi16(uint32_t a, uint32_t k, uint32_t c) {
  uint32_t r;
  asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(a), "s"(k), "v"(c));
  return r;
}

// The largest of three low halves (in the low half).
__device__ __forceinline__ uint32_t max3_u16(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_max3_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Words of a row of the LDS histogram: 256 16-bit or 128 32-bit counters, and 8
// more between the 32-bit rows.  Rows of 128 words put a column's counters of all
// rows into one bank: with 2 bins per axis the lanes met in 2 banks of 64 (820 pairs
// of 300,000 voxels of noise: 528 us, with the 8 words 427), and those of smooth
// fields, which lie along the diagonal, in fewer than now (5,050 pairs of 100,000
// voxels, 128 bins: 757 us, 581).
template <bool PACK16>
constexpr int kRowWords = PACK16 ? 128 : 136;
// ... with H bins per axis (16-bit counters past 128)
inline int row_words(int H) { return H > 128 ? kRowWords<true> : kRowWords<false>; }

// Joint bins of a pair of fields with range [mn, mx] and H <= 256 bins, as
// the reference computes them (JointHistogram.cu:63-75, :127-129): step =
// (mx - mn) / H, bin = (int)((v - mn) / step) clamped to H - 1, step == 0 ->
// bin 0.
//
// Fixed point: z = RN(v R + RN(-mn R - M)), R = 2^16 RN(1 / step), and u =
// floor(z), negative -> 0; u's high half is the bin.  Against 2^16 times the
// reference's quotient RN(RN(v - mn) / step), in units of u: R is off by H 2^-8
// at most over v - mn, the constant's rounding by H 2^-12 (where |mn| / step <=
// H / 16), z's by H 2^-8, the reference's two by H 2^-8 each; z + M is at most
// E = (4 + 1/16) H 2^-8 (1 + 2^-20) off, and M = floor(4 1/8 H 2^-8) + 1 > E.
// Where u's low half is below 2^16 - 2 M the quotient lies inside the interval
// of u's high half, which is therefore the reference's bin; a negative z is a
// quotient below M + E, bin 0.  A quotient at or past H leaves z at most 2 M
// below a multiple of 2^16, so no clamp is needed.  The rare pairs of values
// past that bound (2 x 10 of 65,536 at 256 bins) take the IEEE division; step
// == 0 gives R = 0 and bin 0; a step whose reciprocal is out of range makes
// every pair rare.  Fields far from 0 (|mn| / step > H / 16) subtract first: z =
// RN(RN(v - mn) R - M), with a smaller error.
//
// A pair of values takes two multiply-adds, two conversions, a maximum of the
// low halves (tested once per step) and the address: 7 vector instructions with
// 32-bit counters, 10 with 16-bit ones, at 4 cycles per wave each (31 before,
// by quotients tested one by one for being near an integer).
template <bool PACK16>
struct PairBins {
  float mn, step, r, nm;  // nm: the constant (the subtracting form's: -M)
  uint32_t top;           // largest low half on the fast path
  int hm1;
  bool subtract;

  __device__ __forceinline__ void init(float mn_, float mx_, int H) {
    mn = mn_;
    hm1 = H - 1;
    step = (mx_ - mn_) / (float)H;
    const float q = 1.0f / step;
    const int m = 33 * H / 2048 + 1;
    top = (uint32_t)(65535 - 2 * m);
    r = q * 65536.0f;
    subtract = !(fabsf(mn) * q <= (float)H * 0.0625f);
    nm = subtract ? -(float)m : __builtin_fmaf(-mn, r, -(float)m);
    if (step == 0.0f) {
      r = 0.0f;
      nm = -1.0f;
      subtract = true;
    } else if (!(q < 1e30f && q > 0.0f)) {
      r = 0.0f;
      nm = 65535.0f;
      subtract = true;
    }
  }

  // (a value below mn or a NaN gives bin 0).  The empty statement keeps the
  // division from being carried out ahead of the branch that asks for it.
  __device__ __forceinline__ uint32_t exact(float v) const {
    float a = v - mn;
    asm volatile("" : "+v"(a));
    return (uint32_t)max(min((int)(a / step), hm1), 0);
  }

  // Byte offset of (row, col)'s counter in the LDS histogram.  16-bit counters:
  // 2 per column; bits 0 and 1 are not part of the word's address.  32-bit ones: 4
  // per column.
  static constexpr uint32_t kColBytes = PACK16 ? 2u : 4u;

  // at[u] = offset of (x[u], y[u])'s counter
  template <bool SUB, int N>
  __device__ __forceinline__ void offsets(const float (&x)[N], const float (&y)[N],
                                          uint32_t (&at)[N]) const {
    uint32_t most = 0u;
    auto fixed = [&](float v) {
      return floor_u32(__builtin_fmaf(SUB ? v - mn : v, r, nm));
    };
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const uint32_t ux = fixed(x[u]), uy = fixed(y[u]);
      at[u] = mad_hi16(uy, kColBytes, mad_hi16(ux, 4u * kRowWords<PACK16>, 0u));
      most = max3_u16(most, ux, uy);
    }
    if (__builtin_expect(__ballot((most & 0xffffu) > top) != 0ull, 0)) {
#pragma unroll
      for (int u = 0; u < N; ++u) {
        float a = x[u], b = y[u];
        asm volatile("" : "+v"(a), "+v"(b));  // nothing of this ahead of the branch
        const uint32_t low = max3_u16(0u, fixed(a), fixed(b));
        if (__ballot((low & 0xffffu) > top) != 0ull) at[u] = exact(a) * (4u * kRowWords<PACK16>) + exact(b) * kColBytes;
      }
    }
  }

  // Adds one to the counter at an offset; its word before.
  static __device__ __forceinline__ uint32_t count(uint32_t *s_hist, uint32_t at) {
    char *p = reinterpret_cast<char *>(s_hist);
    if (PACK16)
      return atomicAdd(reinterpret_cast<uint32_t *>(p + (at & ~3u)), 1u << ((at << 3) & 31u));
    return atomicAdd(reinterpret_cast<uint32_t *>(p + at), 1u);
  }
};

// The count of bin (i, j) in the LDS histogram.
template <bool PACK16>
__device__ __forceinline__ uint32_t lds_count(const uint32_t *s, int i, int j) {
  if (PACK16) return (s[i * kRowWords<true> + (j >> 1)] >> ((j & 1) << 4)) & 0xffffu;
  return s[i * kRowWords<false> + j];
}

// word 3 of a raw 32-bit buffer resource on the gfx9 family
constexpr int kBufferWord3 = 0x00020000;

constexpr int kHistBlock = 1024;  // lanes of the histogram workgroups
constexpr int kHistWaves = kHistBlock / 64;

// Which voxel of a step value u of a lane is: a wave takes 64 VPT consecutive
// voxels, a lane 4 consecutive ones of every 256.  Lanes 4 voxels apart meet in
// the same counter less often than neighbours (which an atomic serves one after
// the other), and 4 values arrive per load.
template <int VPT>
__device__ __forceinline__ int voxel_of(int u) {
  static_assert(VPT % 4 == 0, "whole loads");
  return (int)(threadIdx.x >> 6) * 64 * VPT + (u >> 2) * 256 + 4 * (int)(threadIdx.x & 63) + (u & 3);
}

// Voxels of a slice at most: byte offsets into it stay below 2^31.
constexpr int64_t kMaxSlice = (int64_t)1 << 28;

// A slice of a field as a buffer resource whose record count is the slice's
// (at most kMaxSlice voxels, 4-byte aligned): a step is one scalar offset for
// all its loads.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rsrc(const float *f, int len) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(f), 0, 4 * len, kBufferWord3);
}

// A step's values of one slice, from its voxel b on.  A step that reaches past
// the slice's end loads value by value (one past it reads as 0 without a memory
// access).
template <int VPT>
__device__ __forceinline__ void load_values(__amdgpu_buffer_rsrc_t f, int b, int len,
                                            float (&v)[VPT]) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  if (b + kHistBlock * VPT <= len) {
#pragma unroll
    for (int u = 0; u < VPT; u += 4) {
      const u32x4 q = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(f, 4 * voxel_of<VPT>(u), 4 * b, 0));
#pragma unroll
      for (int c = 0; c < 4; ++c) v[u + c] = __uint_as_float(q[c]);
    }
  } else {
    const int at = b < len ? b : len;  // past the end: no record there
#pragma unroll
    for (int u = 0; u < VPT; ++u)
      v[u] = __uint_as_float(
          __builtin_amdgcn_raw_buffer_load_b32(f, 4 * voxel_of<VPT>(u), 4 * at, 0));
  }
}

// Joint counts of the len voxels of slices f1 and f2 into the LDS histogram
// (zero on entry; every lane of a 1024-lane workgroup calls it, the last barrier
// is the caller's): 32-bit counters, which cannot wrap within a call.  The next
// step's values load as soon as this step's are binned.
template <bool SUB, int VPT>
__device__ __attribute__((always_inline)) void accumulate32(const PairBins<false> &bin,
                                                            const float *f1, const float *f2,
                                                            int len, uint32_t *s_hist) {
  constexpr int kStep = kHistBlock * VPT;
  const __amdgpu_buffer_rsrc_t r1 = slice_rsrc(f1, len), r2 = slice_rsrc(f2, len);
  float x[VPT], y[VPT];
  load_values(r1, 0, len, x);
  load_values(r2, 0, len, y);
  for (int b = 0; b < len; b += kStep) {
    uint32_t at[VPT];
    bin.template offsets<SUB>(x, y, at);
    load_values(r1, b + kStep, len, x);
    load_values(r2, b + kStep, len, y);
    if (b + kStep <= len) {
#pragma unroll
      for (int u = 0; u < VPT; ++u) bin.count(s_hist, at[u]);
    } else {
#pragma unroll
      for (int u = 0; u < VPT; ++u)
        if (voxel_of<VPT>(u) < len - b) bin.count(s_hist, at[u]);
    }
  }
}

// The same with 16-bit counters, two to a word.  The lane whose increment finds
// exactly 32,768 in its counter takes them away again and calls rollover(row,
// col) for them, so each passage of that count is answered for once.
//
// No counter wraps: a wave takes round q (8 values per lane) only once every
// wave has answered for round q - 2.  s_prog[q & 1], zero on entry, counts the
// waves' answered rounds of that parity, and a wave adds to it for round q only
// after all have for q - 2, so the sum tells.  While a passage in round r waits
// for its answer no wave is past round r + 1, and when r began every wave had
// answered for r - 2, so fewer than 3 x 8,192 increments follow it: the counter
// stays below 32,768 + 24,576 + 1.  The wave furthest behind never waits, so
// every wait ends.
//
// Barriers in their place cost more: one every 16 values per lane kept the
// waves in step, so that their binning and their atomics took turns, and a
// search for the largest count every 50,000 voxels took 2.5 us each time
// (600x248x248 front, 100 isovalues, 256 bins: counting alone 1.97 ms either
// way, the vector units idle for a third of it).
//
// LOADS rounds of values are on their way at any time.
template <bool SUB, int LOADS, class Rollover>
__device__ __attribute__((always_inline)) void accumulate16(const PairBins<true> &bin,
                                                            const float *f1, const float *f2,
                                                            int len, uint32_t *s_hist,
                                                            uint32_t *s_prog,
                                                            Rollover rollover) {
  constexpr int kVpt = 8, kRound = kHistBlock * kVpt;
  constexpr uint32_t kRoll = 32768u;
  const __amdgpu_buffer_rsrc_t r1 = slice_rsrc(f1, len), r2 = slice_rsrc(f2, len);
  float x[LOADS][kVpt], y[LOADS][kVpt];
#pragma unroll
  for (int r = 0; r < LOADS; ++r) {
    load_values(r1, r * kRound, len, x[r]);
    load_values(r2, r * kRound, len, y[r]);
  }
  auto progress = [&](uint32_t q) -> uint32_t {
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(&s_prog[q & 1u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  };
  auto round = [&](float (&xr)[kVpt], float (&yr)[kVpt], int base, uint32_t q) {
    const uint32_t need = q / 2u * (uint32_t)kHistWaves;
    uint32_t seen = progress(q);
    uint32_t at[kVpt], old[kVpt];
    bin.template offsets<SUB>(xr, yr, at);
    load_values(r1, base + LOADS * kRound, len, xr);
    load_values(r2, base + LOADS * kRound, len, yr);
    while (seen < need) {
      __builtin_amdgcn_s_sleep(1);
      seen = progress(q);
    }
    if (base + kRound <= len) {
#pragma unroll
      for (int u = 0; u < kVpt; ++u) old[u] = bin.count(s_hist, at[u]);
    } else {
#pragma unroll
      for (int u = 0; u < kVpt; ++u)
        old[u] = voxel_of<kVpt>(u) < len - base ? bin.count(s_hist, at[u]) : 0u;
    }
    uint32_t most = 0u;
#pragma unroll
    for (int u = 0; u < kVpt; ++u) most = pk_max_u16(most, old[u]);
    if (__builtin_expect(__ballot((most & (kRoll << 16 | kRoll)) != 0u) != 0ull, 0)) {
#pragma unroll
      for (int u = 0; u < kVpt; ++u) {
        const uint32_t sh = (at[u] << 3) & 31u;
        if (((old[u] >> sh) & 0xffffu) == kRoll) {
          atomicSub(&s_hist[at[u] >> 2], kRoll << sh);
          rollover((int)(at[u] >> 9), (int)((at[u] >> 1) & 255u));
        }
      }
    }
    // relaxed: LDS operations of a wave are carried out in order
    if ((threadIdx.x & 63) == 0)
      __hip_atomic_fetch_add(&s_prog[q & 1u], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  uint32_t q = 0u;
  for (int base = 0; base < len; base += LOADS * kRound) {
#pragma unroll
    for (int r = 0; r < LOADS; ++r) {
      if (r > 0 && base + r * kRound >= len) break;
      round(x[r], y[r], base + r * kRound, q++);
    }
  }
}

// Every lane's share of clearing the first `words` words (a multiple of 4) of
// the LDS histogram.
__device__ __forceinline__ void clear_hist(uint32_t *s_hist, int words) {
  uint4 *p = reinterpret_cast<uint4 *>(s_hist);
  for (int w = threadIdx.x; w < words / 4; w += kHistBlock) p[w] = make_uint4(0u, 0u, 0u, 0u);
}

}  // namespace iso
