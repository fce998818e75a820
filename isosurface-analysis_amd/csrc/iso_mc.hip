// Surface extraction: marching cubes (unique vertices) and the reference's
// voxel approximation, for one or many isovalues per pass over the volume.
//
// Reference semantics, marching cubes (isosurfaces_cuda/src/MarchingCube.cu,
// MarchingCube.cpp:588-710, thrustWrapper.cu:44-56):
//   every classified cell (cube index bit k = corner k < iso, corners clamped
//   to the grid) emits, for every crossed edge, lerp(v_a, v_b, t) with
//   t = (iso - f_a)/(f_b - f_a) in the cell's own edge orientation; the
//   vertex list is sorted and exact duplicates are removed.
//
// MI355X design -- one lane per grid point P, owning the three edges
// P->P+e_x, P->P+e_y, P->P+e_z:
//   - a vertex whose along-edge coordinate is not an integer lies strictly
//     inside its grid edge, so it can only coincide with vertices of the same
//     edge; those come in two orientations (+ from cells on one side, - from
//     the other), so deduplication is a compare of at most two values, done
//     in registers by the edge's owner;
//   - a vertex that lands exactly on a grid point (t rounds to 0 or 1, or a
//     sample equals iso) can coincide across edges; it is inserted into a
//     hash set keyed by (isovalue, grid point) and emitted by the winner;
//   - which orientations exist depends only on which cells contain the edge
//     (grid extent and the reference's classify limit), computed once;
//   - the workgroup loops over only the isovalues inside the [min,max] of its
//     samples (block culling), so one read of the volume serves all k
//     isovalues of an ISM;
//   - a count pass and a scan give every (block, isovalue, wave) its place in
//     the output; the vertex set is exact, its order unspecified.
#include "iso_internal.hpp"

#include <algorithm>
#include <cstring>
#include <numeric>
#include <type_traits>
#include <vector>

namespace iso {
int exclusive_scan_u32(iso_ctx *ctx, const uint32_t *d_in, uint32_t *d_out, int64_t n,
                       uint32_t *d_total, uint32_t *d_tmp);
size_t scan_tmp_words(int64_t n);
int radix_sort_pairs(iso_ctx *ctx, uint32_t **keys, uint32_t **vals, uint32_t *keys_alt,
                     uint32_t *vals_alt, int64_t n, int bits);
int iota_u32(iso_ctx *ctx, uint32_t *d, int64_t n);
}  // namespace iso

namespace {

constexpr int kMcBlock = 256;
constexpr int kMcWaves = kMcBlock / 64;
constexpr int kMcRound = 32;  // isovalues per pool reservation (bit masks of 32)
constexpr unsigned long long kEmpty = ~0ull;
constexpr int kMcOddVertices = 4;  // word of the counters

// ---- case tables, generated from first principles -------------------------
// Corners 0..7 of a cell sit at (0,0,0) (1,0,0) (1,1,0) (0,1,0) (0,0,1)
// (1,0,1) (1,1,1) (0,1,1); edge e joins kEdge[e][0] -> kEdge[e][1] (the
// reference's numbering, MarchingCube.cu:208-265).  A case's vertex count is
// 3*(#crossed edges - 2*#polygons); polygons join crossed edges face by face,
// cutting off the corners below iso on faces with four crossed edges.
const int kEdge[12][2] = {{0, 1}, {1, 2}, {2, 3}, {3, 0}, {4, 5}, {5, 6},
                          {6, 7}, {7, 4}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};
const int kFace[6][4] = {{0, 1, 2, 3}, {4, 5, 6, 7}, {0, 1, 5, 4},
                         {1, 2, 6, 5}, {2, 3, 7, 6}, {3, 0, 4, 7}};

int find_root(int *p, int x) {
  while (p[x] != x) x = p[x] = p[p[x]];
  return x;
}

struct CaseTables {
  uint8_t nverts[256];
  CaseTables() {
    for (int c = 0; c < 256; ++c) {
      int crossed = 0, ne = 0, parent[12];
      for (int e = 0; e < 12; ++e) {
        parent[e] = e;
        if (((c >> kEdge[e][0]) & 1) != ((c >> kEdge[e][1]) & 1)) { crossed |= 1 << e; ++ne; }
      }
      for (int f = 0; f < 6; ++f) {
        int fe[4], ce[4], nc = 0;
        for (int i = 0; i < 4; ++i) {
          int a = kFace[f][i], b = kFace[f][(i + 1) & 3];
          for (int e = 0; e < 12; ++e)
            if ((kEdge[e][0] == a && kEdge[e][1] == b) || (kEdge[e][0] == b && kEdge[e][1] == a))
              fe[i] = e;
          if (crossed >> fe[i] & 1) ce[nc++] = fe[i];
        }
        if (nc == 2) parent[find_root(parent, ce[0])] = find_root(parent, ce[1]);
        if (nc == 4)
          for (int i = 0; i < 4; ++i)
            if ((c >> kFace[f][i]) & 1)
              parent[find_root(parent, fe[(i + 3) & 3])] = find_root(parent, fe[i]);
      }
      int polys = 0;
      for (int e = 0; e < 12; ++e)
        if ((crossed >> e & 1) && find_root(parent, e) == e) ++polys;
      nverts[c] = (uint8_t)(3 * (ne - 2 * polys));
    }
  }
};

const CaseTables &case_tables() {
  static CaseTables t;
  return t;
}

struct McArgs {
  const float *vol;
  int gx, gy, gz;          // sample extent per logical axis (corner clamp)
  int64_t sx, sy, sz;      // element strides of logical x, y, z
  int ncx, ncy, ncz;       // cells per axis
  int npx, npy, npz;       // grid points per axis (ncells + 1)
  int64_t npoints;
  int64_t ncls;            // cells with linear index x + gx*(y + gy*z) below this are classified
  int zfast;               // lane order: z fastest (1) or x fastest (0)
  const float *isos;       // ascending
  const int *slot;         // sorted index -> caller's isovalue index
  int k;
  uint32_t *counts;        // per slot: vertices found
  unsigned long long *stats;  // per slot: active cells, total vertices
  float *out;              // vertex pool, xyz triples (all isovalues, any order)
  uint32_t *out_slot;      // per pool vertex: isovalue slot (may be null)
  int64_t cap;             // pool capacity in vertices (0 = count only)
  unsigned long long *corner_tab;
  uint32_t *corner_owner;  // per table slot: id of the candidate that inserted the key
  uint32_t corner_mask;
  uint32_t *overflow;
  uint32_t *block_total;       // count pass: vertices per block
  const uint32_t *block_base;  // emit pass: exclusive scan of block_total
  // vertices per (isovalue of a round, wave) of each block (at most 64 x 5,
  // 16 bits), written by the count pass and read by the emit pass:
  // max_rounds x kMcRound x kMcWaves entries per block
  uint16_t *wave_counts;
  int max_rounds;
  uint32_t *counts_priv;       // [kMcPriv][k] vertices per slot, privatised
  unsigned long long *stats_priv;  // [kMcPriv][2k] active cells, case vertices
  uint8_t nverts[256];
};

constexpr int kMcPriv = 64;   // copies of the per-slot counters (blocks spread over them)

__device__ __forceinline__ uint64_t hash64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Count pass: true if this candidate inserted the key (first claim of a
// grid-point vertex); the inserter records its id beside the key.
__device__ __forceinline__ bool corner_claim(const McArgs &a, uint64_t key, uint32_t id) {
  uint32_t h = (uint32_t)hash64(key) & a.corner_mask;
  for (int probe = 0; probe < 128; ++probe) {
    unsigned long long old = atomicCAS(&a.corner_tab[h], kEmpty, (unsigned long long)key);
    if (old == kEmpty) {
      a.corner_owner[h] = id;
      return true;
    }
    if (old == key) return false;
    h = (h + 1) & a.corner_mask;
  }
  atomicAdd(a.overflow, 1u);  // table too full: the host retries with a larger one
  return false;
}

// Emit pass (a later launch): true if this candidate inserted the key.
__device__ __forceinline__ bool corner_owned(const McArgs &a, uint64_t key, uint32_t id) {
  uint32_t h = (uint32_t)hash64(key) & a.corner_mask;
  for (int probe = 0; probe < 128; ++probe) {
    const unsigned long long k = a.corner_tab[h];
    if (k == key) return a.corner_owner[h] == id;
    if (k == kEmpty) return false;
    h = (h + 1) & a.corner_mask;
  }
  return false;
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

// number of set bits of m in lanes below this one
__device__ __forceinline__ uint32_t lane_prefix(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ bool cell_ok(const McArgs &a, int cx, int cy, int cz) {
  if (cx < 0 || cy < 0 || cz < 0 || cx >= a.ncx || cy >= a.ncy || cz >= a.ncz) return false;
  int64_t lin = (int64_t)cx + (int64_t)a.gx * ((int64_t)cy + (int64_t)a.gy * cz);
  return lin < a.ncls;
}

// f over the lanes of the wave: rotations within rows of 16, then the lanes 16
// and 32 away
template <class F>
__device__ __forceinline__ float wave_fold(float v, F f) {
  auto rot = [](float x, auto r) {
    const int i = __float_as_int(x);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x120 + decltype(r)::value, 0xf, 0xf, true));
  };
  v = f(v, rot(v, std::integral_constant<int, 1>()));
  v = f(v, rot(v, std::integral_constant<int, 2>()));
  v = f(v, rot(v, std::integral_constant<int, 4>()));
  v = f(v, rot(v, std::integral_constant<int, 8>()));
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(p[0]), __uint_as_float(p[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

__device__ __forceinline__ void wave_minmax(float &lo, float &hi) {
  lo = wave_fold(lo, [](float a, float b) { return fminf(a, b); });
  hi = wave_fold(hi, [](float a, float b) { return fmaxf(a, b); });
}

// isovalues that values in [lo, hi] can cross, lo < iso <= hi: [first, second)
// (a NaN, which nothing crosses, stands past all others and counts in neither)
__device__ __forceinline__ int2 iso_range(const float *isos, int k, float lo, float hi) {
  int b0 = 0, b1 = 0;
  for (int i = threadIdx.x & 63; __ballot(i < k); i += 64) {
    const float v = i < k ? isos[i] : 0.0f;
    b0 += __popcll(__ballot(i < k && v <= lo));
    b1 += __popcll(__ballot(i < k && v <= hi));
  }
  return make_int2(b0, lo <= hi ? b1 : b0);
}

// exclusive prefix sum over the first 32 lanes, and their sum
__device__ __forceinline__ uint32_t prefix32(uint32_t v, uint32_t &sum) {
  const int lane = threadIdx.x & 63;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  sum = (uint32_t)__builtin_amdgcn_readlane((int)inc, 31);
  return inc - v;
}

constexpr int kMcF = 17, kMcM = 5;  // samples of a block: 16 x 4 x 4 and one more per axis
constexpr int kMcQueue = 256;       // crossings of a wave waiting to be worked out

// EMIT = false: count pass (claims grid-point vertices, per-block totals,
// per-slot counts and, when STATS, cell statistics).  EMIT = true: the same
// decisions again, grid-point vertices taken by their recorded owner,
// vertices written from the block's scanned base.  No pool counter is shared
// between blocks.
//
// A wave goes over its isovalues with one compare per sample: a crossing of a
// lane's edge is a bit where two masks differ, and the crossings go into the
// wave's queue, isovalue by isovalue.  64 at a time they are worked out with
// every lane busy (divisions, orientations, grid points).  Most lanes of a wave
// cross no given isovalue, so working the edges out isovalue by isovalue ran
// the divisions of all five candidates for a few lanes each.
// Bound by the vector instructions (3.7 cycles each): the queueing about half
// of them, the working out a third, the rest the block's start.  418M vertices
// of 64 isovalues over 512^3 sines: count 6.6 -> 4.0 ms, emit 9.1 -> 4.1 (6.7 GB
// written, 1.6 TB/s); 174M of 100 over the 600x248x248 front: 1.17 -> 0.98 and
// 1.63 -> 1.21; one isovalue of the front 340 -> 238 and 298 -> 66 us (blocks
// without a vertex leave at once).  Several blocks per workgroup with the next
// one's samples under way (2, 4, 8): front 2.38, sines 8.7 ms, no gain.
// A vertex's place is its number in the wave's order plus, per isovalue, what
// turns that order (wave, isovalue) into the block's (isovalue, wave), so that
// an isovalue's vertices of a block are one run of the pool.
template <bool EMIT, bool STATS>
__global__ __launch_bounds__(kMcBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void mc_kernel(McArgs a) {
  __shared__ float s_v[kMcF * kMcM * kMcM];
  __shared__ uint32_t s_queue[kMcWaves][kMcQueue];
  __shared__ uint8_t s_nv[256];
  __shared__ float s_lo[kMcWaves], s_hi[kMcWaves];
  __shared__ uint32_t s_nan[kMcWaves];  // count pass: NaN samples
  // count pass, per (isovalue of the round, wave), of two rounds in turn:
  // vertices, active cells, case vertices; corrections to the vertices
  __shared__ uint32_t s_wt[2][kMcRound][kMcWaves], s_wa[2][kMcRound][kMcWaves];
  __shared__ uint32_t s_wv[2][kMcRound][kMcWaves];
  __shared__ int s_fix[kMcWaves][kMcRound];
  __shared__ uint32_t s_run;  // count pass: vertices of the block so far
  if (EMIT && a.block_total[blockIdx.x] == 0u) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (STATS) s_nv[tid] = a.nverts[tid];
  if (!EMIT) {
    if (tid < kMcWaves * kMcRound) (&s_fix[0][0])[tid] = 0;
    if (tid == 0) s_run = 0u;
  }

  // A block owns a brick of 16 x 4 x 4 grid points, 16 along the memory-fast
  // axis (z, or x when zfast is 0): a small brick spans a narrower value range
  // than a 256-point line, so fewer isovalues reach it.
  int px, py, pz;  // the block's first grid point
  {
    const uint32_t nbf = (uint32_t)((a.zfast ? a.npz : a.npx) + 15) >> 4;
    const uint32_t nby = (uint32_t)(a.npy + 3) >> 2, b = blockIdx.x;
    const int f = (int)(b % nbf) * 16, m = (int)(b / nbf / nby) * 4;
    py = (int)(b / nbf % nby) * 4;
    px = a.zfast ? m : f;
    pz = a.zfast ? f : m;
  }
  const int ex = a.zfast ? 4 : 16, ez = a.zfast ? 16 : 4;  // the brick's extent
  {
    float lo = 3.4e38f, hi = -3.4e38f;
    bool nan = false;
    const uint32_t sm = (uint32_t)(a.zfast ? a.sx : a.sz), sy = (uint32_t)a.sy;
    const bool inside = px + (a.zfast ? kMcM : kMcF) <= a.gx && py + kMcM <= a.gy &&
                        pz + (a.zfast ? kMcF : kMcM) <= a.gz;
    const float *corner = a.vol + (px * a.sx + py * a.sy + pz * a.sz);
#pragma unroll
    for (uint32_t i = tid; i < kMcF * kMcM * kMcM; i += kMcBlock) {
      const uint32_t row = (i * 241u) >> 12, f = i - row * kMcF;  // i / 17 below 425
      const uint32_t m2 = (row * 205u) >> 10, m1 = row - m2 * kMcM;  // row / 5 below 25
      float v;
      if (inside) {
        v = corner[f + m1 * sy + m2 * sm];  // below 5 / 2 x the grid points in all
      } else {
        const int x = min(px + (int)(a.zfast ? m2 : f), a.gx - 1), y = min(py + (int)m1, a.gy - 1);
        const int z = min(pz + (int)(a.zfast ? f : m2), a.gz - 1);
        v = a.vol[x * a.sx + y * a.sy + z * a.sz];
      }
      s_v[i] = v;
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
      if (!EMIT) nan |= v != v;
    }
    wave_minmax(lo, hi);
    const uint64_t nans = __ballot(nan);
    if (lane == 0) {
      s_lo[w] = lo;
      s_hi[w] = hi;
      if (!EMIT) s_nan[w] = nans != 0ull;
    }
  }
  __syncthreads();
  int j0, j1;
  {
    float lo = s_lo[0], hi = s_hi[0];
#pragma unroll
    for (int q = 1; q < kMcWaves; ++q) { lo = fminf(lo, s_lo[q]); hi = fmaxf(hi, s_hi[q]); }
    const int2 r = iso_range(a.isos, a.k, lo, hi);
    j0 = r.x;
    j1 = r.y;
  }
  if (j0 >= j1) {
    if (!EMIT && tid == 0) a.block_total[blockIdx.x] = 0u;
    return;
  }

  // this lane's grid point, and the steps to its neighbours in s_v
  const int lf = lane & 15, l1 = lane >> 4;
  const int x = px + (a.zfast ? w : lf), y = py + l1, z = pz + (a.zfast ? lf : w);
  const int dx = a.zfast ? kMcF * kMcM : 1, dz = a.zfast ? 1 : kMcF * kMcM;
  const int at = lf + kMcF * l1 + kMcF * kMcM * w;
  const float v0 = s_v[at], vx = s_v[at + dx], vy = s_v[at + kMcF], vz = s_v[at + dz];
  // which cells around P exist and are classified (isovalue independent):
  // all of them, inside
  bool xp = true, xm = true, yp = true, ym = true, zp = true, cell = true;
  if (px == 0 || py == 0 || pz == 0 || px + ex > a.ncx || py + 4 > a.ncy || pz + ez > a.ncz ||
      px + ex - 1 + (int64_t)a.gx * (py + 3 + (int64_t)a.gy * (pz + ez - 1)) >= a.ncls) {
    const bool live = x < a.npx && y < a.npy && z < a.npz;
    const bool c000 = live && cell_ok(a, x, y, z);
    const bool c001 = live && cell_ok(a, x, y, z - 1);
    const bool c010 = live && cell_ok(a, x, y - 1, z);
    const bool c011 = live && cell_ok(a, x, y - 1, z - 1);
    const bool c100 = live && cell_ok(a, x - 1, y, z);
    const bool c101 = live && cell_ok(a, x - 1, y, z - 1);
    const bool c110 = live && cell_ok(a, x - 1, y - 1, z);
    xp = c000 || c001;  // x edge: + / - orientation present
    xm = c010 || c011;
    yp = c100 || c101;  // y edge
    ym = c000 || c001;
    zp = c000 || c100 || c010 || c110;  // z edge (always +)
    cell = c000;
  }
  const uint64_t has_x = __ballot(xp || xm), has_y = __ballot(yp || ym), has_z = __ballot(zp);
  // a crossing: lane | edge << 6 | + present << 8 | - present << 9 | isovalue << 10
  const uint32_t item_x = lane | (uint32_t)xp << 8 | (uint32_t)xm << 9;
  const uint32_t item_y = lane | 1u << 6 | (uint32_t)yp << 8 | (uint32_t)ym << 9;
  const uint32_t item_z = lane | 2u << 6 | 1u << 8;
  // the isovalues this wave's edges can cross
  int2 own = make_int2(j0, j1);
  // With NaN samples in the block, a wave looks at an isovalue if one of its
  // cells has a corner below it and one at or above it, NaN corners aside, and
  // then takes every edge whose ends compare differently, an edge to a NaN
  // among them.  (Without NaN samples this is what the crossings give: an edge
  // that crosses an isovalue is an edge of such a cell.)
  const bool nans = !EMIT && (s_nan[0] | s_nan[1] | s_nan[2] | s_nan[3]) != 0u;
  static_assert(kMcWaves == 4, "four flags");
  if (!EMIT && !STATS && !nans) {
    float lo = fminf(fminf(v0, vx), fminf(vy, vz)), hi = fmaxf(fmaxf(v0, vx), fmaxf(vy, vz));
    wave_minmax(lo, hi);
    own = iso_range(a.isos, a.k, lo, hi);
  }
  const int64_t bbase = EMIT ? (int64_t)a.block_base[blockIdx.x] : 0;
  float *const out = a.out + 3 * bbase;
  uint32_t *const out_slot = a.out_slot ? a.out_slot + bbase : nullptr;
  const uint32_t room = EMIT ? (uint32_t)min(max(a.cap - bbase, (int64_t)0), (int64_t)INT32_MAX) : 0u;
  uint32_t run = 0;  // emit pass: vertices of the block in the rounds before
  for (int jc = j0, round = 0; jc < j1; jc += kMcRound, ++round) {
    const int jn = min(kMcRound, j1 - jc);
    uint16_t *wc = a.wave_counts + ((int64_t)blockIdx.x * a.max_rounds + round) *
                                       (kMcRound * kMcWaves);
    // lane u holds isovalue u of the round
    const float iso_u = lane < jn ? a.isos[jc + lane] : 0.0f;
    const int slot_u = lane < jn ? a.slot[jc + lane] : 0;
    uint32_t count_u = 0, rel_u = 0;
    uint64_t todo;  // the isovalues to look at
    if (EMIT) {
      // the vertices of the round's isovalues in each wave from the count pass
      ushort4 c = make_ushort4(0, 0, 0, 0);
      if (lane < jn) c = ((const ushort4 *)wc)[lane];
      const uint32_t mine = w == 0 ? c.x : w == 1 ? c.y : w == 2 ? c.z : c.w;
      const uint32_t before = (w > 0 ? c.x : 0) + (w > 1 ? c.y : 0) + (w > 2 ? c.z : 0);
      uint32_t all, ours;
      rel_u = run + before + prefix32(c.x + c.y + c.z + c.w, all) - prefix32(mine, ours);
      run += all;
      todo = __ballot(mine != 0u);
    } else {
      const int u0 = max(own.x - jc, 0), u1 = min(own.y - jc, jn);
      todo = u1 > u0 ? (~0ull >> (64 - u1)) & (~0ull << u0) : 0ull;
      if (nans) {
        float lo = 3.4e38f, hi = -3.4e38f;
        if (__builtin_amdgcn_inverse_ballot_w64(has_x | has_y | has_z)) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const float v = s_v[at + (q & 1 ? dx : 0) + (q & 2 ? kMcF : 0) + (q & 4 ? dz : 0)];
            lo = fminf(lo, v);
            hi = fmaxf(hi, v);
          }
        }
        uint64_t reached = 0ull;
        for (uint64_t t = todo; t; t &= t - 1) {
          const int u = __ffsll((unsigned long long)t) - 1;
          const float iso = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(iso_u), u));
          if (__ballot(lo < iso && iso <= hi)) reached |= 1ull << u;
        }
        if (STATS && lane < jn)
          s_wa[round & 1][lane][w] = s_wv[round & 1][lane][w] = 0u;  // of those left out
        todo = reached;
      }
    }
    uint32_t head = 0, tail = 0, seq = 0;
    // works out the n crossings at the queue's head, one per lane
    auto work_out = [&](uint32_t n) {
      const uint32_t item = s_queue[w][(head + lane) & (kMcQueue - 1)];
      const bool valid = (uint32_t)lane < n;
      const int l = item & 63, edge = (item >> 6) & 3, u = (item >> 10) & 31;
      const bool plus = item & (1u << 8), minus = item & (1u << 9);
      const int qf = l & 15, q1 = (l >> 4) & 3;
      const int qx = px + (a.zfast ? w : qf), qy = py + q1, qz = pz + (a.zfast ? qf : w);
      const int p0 = qf + kMcF * q1 + kMcF * kMcM * w;
      const float f0 = s_v[p0], f1 = s_v[p0 + (edge == 0 ? dx : edge == 1 ? kMcF : dz)];
      const float iso = __int_as_float(__builtin_amdgcn_ds_bpermute(u << 2, __float_as_int(iso_u)));
      const float fx = (float)qx, fy = (float)qy, fz = (float)qz;
      const float base = edge == 0 ? fx : edge == 1 ? fy : fz;
      const float vp = base + (iso - f0) / (f1 - f0);
      const float vm = (base + 1.0f) - (iso - f1) / (f0 - f1);
      bool has_p = valid && plus, has_m = valid && minus && !(plus && vp == vm);
      // grid-point vertices: the first claim wins (count pass), its owner emits
      const bool grid_p = has_p && (vp == base || vp == base + 1.0f);
      const bool grid_m = has_m && (vm == base || vm == base + 1.0f);
      int slot = 0;
      if (EMIT || __ballot(grid_p || grid_m)) slot = __builtin_amdgcn_ds_bpermute(u << 2, slot_u);
      if (grid_p || grid_m) {
        const uint32_t id =
            (uint32_t)(((int64_t)qz * a.npy + qy) * a.npx + qx) * 5u + 2u * (uint32_t)edge;
        auto take = [&](float v, uint32_t kind) {
          const int gx = edge == 0 ? (int)v : qx, gy = edge == 1 ? (int)v : qy;
          const int gz = edge == 2 ? (int)v : qz;
          const uint64_t key =
              (uint64_t)slot << 40 |
              (uint64_t)((int64_t)gx + (int64_t)a.npx * ((int64_t)gy + (int64_t)a.npy * gz));
          return EMIT ? corner_owned(a, key, id + kind) : corner_claim(a, key, id + kind);
        };
        if (grid_p) has_p = take(vp, 0u);
        if (grid_m) has_m = take(vm, 1u);
      }
      if (EMIT) {
        const uint64_t bp = __ballot(has_p), bm = __ballot(has_m);
        const uint32_t rel = (uint32_t)__builtin_amdgcn_ds_bpermute(u << 2, (int)rel_u);
        uint32_t pos = rel + seq + lane_prefix(bp) + lane_prefix(bm);
        seq += (uint32_t)__popcll(bp) + (uint32_t)__popcll(bm);
        auto put = [&](float v) {
          if (pos < room) {
            float3 p;
            p.x = edge == 0 ? v : fx;
            p.y = edge == 1 ? v : fy;
            p.z = edge == 2 ? v : fz;
            *(float3 *)(out + 3u * pos) = p;
            if (out_slot) out_slot[pos] = (uint32_t)slot;
          }
          ++pos;
        };
        if (has_p) put(vp);
        if (has_m) put(vm);
      } else {  // one vertex has been counted for it
        const int fix = (int)has_p + (int)has_m - 1;
        if (valid && fix) atomicAdd(&s_fix[w][u], fix);
      }
      head += n;
    };
    while (todo) {
      const int u = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const float iso = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(iso_u), u));
      const uint64_t m0 = __ballot(v0 < iso);
      const uint64_t cx = (m0 ^ __ballot(vx < iso)) & has_x;
      const uint64_t cy = (m0 ^ __ballot(vy < iso)) & has_y;
      const uint64_t cz = (m0 ^ __ballot(vz < iso)) & has_z;
      const uint32_t n = (uint32_t)__popcll(cx) + (uint32_t)__popcll(cy) + (uint32_t)__popcll(cz);
      if (n) {
        // a lane's crossings in a row, lane after lane
        uint32_t r = tail + lane_prefix(cx) + lane_prefix(cy) + lane_prefix(cz);
        const uint32_t tag = (uint32_t)u << 10;
        if (__builtin_amdgcn_inverse_ballot_w64(cx)) s_queue[w][r++ & (kMcQueue - 1)] = item_x | tag;
        if (__builtin_amdgcn_inverse_ballot_w64(cy)) s_queue[w][r++ & (kMcQueue - 1)] = item_y | tag;
        if (__builtin_amdgcn_inverse_ballot_w64(cz)) s_queue[w][r & (kMcQueue - 1)] = item_z | tag;
        tail += n;
        if (!EMIT) count_u = lane == u ? n : count_u;
        while (tail - head >= 64u) work_out(64u);
      }
      if (STATS) {
        // cell statistics of the cell at P, reference corner order
        const float s[8] = {v0,
                            vx,
                            s_v[at + dx + kMcF],
                            vy,
                            vz,
                            s_v[at + dx + dz],
                            s_v[at + dx + kMcF + dz],
                            s_v[at + kMcF + dz]};
        uint32_t ci = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) ci |= (uint32_t)(s[q] < iso) << q;
        const uint32_t tot = cell ? s_nv[ci] : 0u;
        const uint32_t act_w = __popcll(__ballot(tot != 0u));
        const uint32_t tot_w = __popcll(__ballot(tot & 1u)) + 2 * __popcll(__ballot(tot & 2u)) +
                               4 * __popcll(__ballot(tot & 4u)) + 8 * __popcll(__ballot(tot & 8u));
        if (lane == 0) { s_wa[round & 1][u][w] = act_w; s_wv[round & 1][u][w] = tot_w; }
      }
    }
    if (tail != head) work_out(tail - head);
    if (!EMIT) {
      if (lane < jn) {
        s_wt[round & 1][lane][w] = count_u + (uint32_t)s_fix[w][lane];
        s_fix[w][lane] = 0;
      }
      // the waves' counts of a round are read while the next one's go into the
      // other half
      __syncthreads();
      if (tid < jn) {
        const uint32_t *wt = s_wt[round & 1][tid];
        ((ushort4 *)wc)[tid] = make_ushort4((uint16_t)wt[0], (uint16_t)wt[1], (uint16_t)wt[2],
                                            (uint16_t)wt[3]);
        const uint32_t vj = wt[0] + wt[1] + wt[2] + wt[3];
        uint32_t aj = 0, tj = 0;
        if (STATS) {
#pragma unroll
          for (int q = 0; q < kMcWaves; ++q) {
            aj += s_wa[round & 1][tid][q];
            tj += s_wv[round & 1][tid][q];
          }
        }
        const int64_t priv = (int64_t)(blockIdx.x % kMcPriv) * a.k + slot_u;
        if (vj) {
          atomicAdd(&a.counts_priv[priv], vj);
          atomicAdd(&s_run, vj);
        }
        if (STATS && aj) {
          atomicAdd(&a.stats_priv[priv * 2], (unsigned long long)aj);
          atomicAdd(&a.stats_priv[priv * 2 + 1], (unsigned long long)tj);
        }
      }
    }
  }
  // (wave 0 added up the rounds)
  if (!EMIT && tid == 0) a.block_total[blockIdx.x] = s_run;
}

// Per-isovalue totals from the privatised counters (counts[s] = the sum of
// the kMcPriv copies; stats likewise unless stats is null), and their 64-bit
// sum into *total64 (which the 32-bit vertex offsets are checked against).
__global__ void mc_reduce_kernel(const uint32_t *counts_priv, const unsigned long long *stats_priv,
                                 int k, uint32_t *counts, unsigned long long *stats,
                                 unsigned long long *total64) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= k) return;
  uint32_t c = 0;
  unsigned long long a0 = 0, a1 = 0;
  for (int p = 0; p < kMcPriv; ++p) {
    c += counts_priv[(int64_t)p * k + s];
    if (stats) {
      a0 += stats_priv[((int64_t)p * k + s) * 2];
      a1 += stats_priv[((int64_t)p * k + s) * 2 + 1];
    }
  }
  counts[s] = c;
  atomicAdd(total64, (unsigned long long)c);
  if (stats) {
    stats[2 * s] = a0;
    stats[2 * s + 1] = a1;
  }
}

// ---- voxel approximation ----------------------------------------------------
// Cell (x,y,z), x<X-1, y<Y-1, z<Z-1 of the z-fastest image is emitted iff one
// corner is > iso and one is < iso (IsosurfaceApproximation.cu:67-135);
// output order is the cell order x-major / z-fastest (stable copy_if).
constexpr int kApBlock = 256;
constexpr int kApItems = 4;
constexpr int kApTile = kApBlock * kApItems;

struct ApArgs {
  const float *img;
  int X, Y, Z;
  int64_t ncells;
  float iso;
  uint32_t *tile_counts;
  const uint32_t *tile_offsets;
  int32_t *out;
  int64_t cap;
};

__device__ __forceinline__ bool approx_flag(const ApArgs &a, int64_t o) {
  const int64_t Zc = a.Z - 1, Yc = a.Y - 1;
  const int z = (int)(o % Zc);
  const int y = (int)((o / Zc) % Yc);
  const int x = (int)(o / (Zc * Yc));
  const int64_t YZ = (int64_t)a.Y * a.Z;
  const int64_t lu = x * YZ + (int64_t)y * a.Z + z;
  const float *p = a.img + lu;
  const float c[8] = {p[0], p[1], p[a.Z], p[a.Z + 1], p[YZ], p[YZ + 1], p[YZ + a.Z], p[YZ + a.Z + 1]};
  bool above = false, below = false;
#pragma unroll
  for (int q = 0; q < 8; ++q) { above |= c[q] > a.iso; below |= c[q] < a.iso; }
  return above && below;
}

// tile t covers cells [t*kApTile, (t+1)*kApTile), item q of lane l is cell
// t*kApTile + l*kApItems + q (contiguous per lane, so tile order = cell order)
__global__ __launch_bounds__(kApBlock) void approx_count_kernel(ApArgs a) {
  __shared__ uint32_t s_w[kApBlock / 64];
  const int64_t base = (int64_t)blockIdx.x * kApTile + (int64_t)threadIdx.x * kApItems;
  uint32_t c = 0;
#pragma unroll
  for (int q = 0; q < kApItems; ++q)
    if (base + q < a.ncells) c += approx_flag(a, base + q);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kApBlock / 64; ++w) t += s_w[w];
    a.tile_counts[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kApBlock) void approx_emit_kernel(ApArgs a) {
  __shared__ uint32_t s_w[kApBlock / 64];
  const int64_t base = (int64_t)blockIdx.x * kApTile + (int64_t)threadIdx.x * kApItems;
  bool f[kApItems];
  uint32_t c = 0;
#pragma unroll
  for (int q = 0; q < kApItems; ++q) {
    f[q] = base + q < a.ncells && approx_flag(a, base + q);
    c += f[q];
  }
  const uint32_t inc = wave_incl_scan(c);
  if ((threadIdx.x & 63) == 63) s_w[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t wpre = 0;
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) wpre += s_w[w];
  int64_t pos = (int64_t)a.tile_offsets[blockIdx.x] + wpre + inc - c;
  const int64_t Zc = a.Z - 1, Yc = a.Y - 1;
#pragma unroll
  for (int q = 0; q < kApItems; ++q) {
    if (f[q]) {
      if (pos < a.cap) {
        const int64_t o = base + q;
        a.out[3 * pos] = (int32_t)(o / (Zc * Yc));
        a.out[3 * pos + 1] = (int32_t)((o / Zc) % Yc);
        a.out[3 * pos + 2] = (int32_t)(o % Zc);
      }
      ++pos;
    }
  }
}

// Many isovalues per pass (unordered pool output, for the pipeline): lane =
// cell of a 4 x 4 x 16 brick (z fastest), whose samples are staged in LDS once
// (425 for 256 cells), block-culled loop over the isovalues strictly inside the
// block's [min, max] in rounds of 32: pass 1 counts per wave, one pool
// reservation per block and round, pass 2 writes.  Bound by its vector
// instructions and the volume's one reading: 256 isovalues of a
// 200x160x120 volume 640 -> 121 us (eight loads per cell, and one lane that laid
// out a round's 128 places and counted each isovalue, before).
struct ApMultiArgs {
  const float *img;
  int X, Y, Z;
  const float *isos;  // ascending
  const int *slot;
  int k;
  uint32_t *counts;
  int32_t *out;        // pool of xyz cells
  uint32_t *out_slot;  // per pool entry: isovalue slot
  int64_t cap;
  unsigned long long *pool_count;
};

constexpr int kApWaves = kApBlock / 64;
constexpr int kApRound = 32;

__global__ __launch_bounds__(kApBlock) void approx_multi_kernel(ApMultiArgs a) {
  __shared__ float s_v[kMcF * kMcM * kMcM];  // the block's samples, one more per axis
  __shared__ float s_lo[kApWaves], s_hi[kApWaves];
  __shared__ uint32_t s_wt[kApRound][kApWaves], s_off[kApRound][kApWaves];
  __shared__ unsigned long long s_base;
  __shared__ uint32_t s_run;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int Xc = a.X - 1, Yc = a.Y - 1, Zc = a.Z - 1;
  const uint32_t nbz = (uint32_t)(Zc + 15) >> 4, nby = (uint32_t)(Yc + 3) >> 2, b = blockIdx.x;
  const int z0 = (int)(b % nbz) * 16, y0 = (int)(b / nbz % nby) * 4, x0 = (int)(b / nbz / nby) * 4;
  const int64_t YZ = (int64_t)a.Y * a.Z;
  for (uint32_t i = tid; i < kMcF * kMcM * kMcM; i += kApBlock) {
    const uint32_t row = (i * 241u) >> 12, f = i - row * kMcF;     // i / 17 below 425
    const uint32_t m2 = (row * 205u) >> 10, m1 = row - m2 * kMcM;  // row / 5 below 25
    const int x = min(x0 + (int)m2, a.X - 1), y = min(y0 + (int)m1, a.Y - 1);
    s_v[i] = a.img[x * YZ + (int64_t)y * a.Z + min(z0 + (int)f, a.Z - 1)];
  }
  __syncthreads();
  const int lf = lane & 15, l1 = lane >> 4;
  const int x = x0 + w, y = y0 + l1, z = z0 + lf;
  float lo = 3.4e38f, hi = -3.4e38f;
  if (x < Xc && y < Yc && z < Zc) {
    const float *p = s_v + lf + kMcF * l1 + kMcF * kMcM * w;
    constexpr int dy = kMcF, dx = kMcF * kMcM;
    const float c[8] = {p[0], p[1], p[dy], p[dy + 1], p[dx], p[dx + 1], p[dx + dy], p[dx + dy + 1]};
#pragma unroll
    for (int q = 0; q < 8; ++q) { lo = fminf(lo, c[q]); hi = fmaxf(hi, c[q]); }
  }
  {
    float wlo = lo, whi = hi;
    wave_minmax(wlo, whi);
    if (lane == 0) { s_lo[w] = wlo; s_hi[w] = whi; }
  }
  __syncthreads();
  int j0 = 0, j1 = 0;  // the isovalues strictly inside the block's range
  {
    float L = s_lo[0], Hh = s_hi[0];
#pragma unroll
    for (int q = 1; q < kApWaves; ++q) { L = fminf(L, s_lo[q]); Hh = fmaxf(Hh, s_hi[q]); }
    for (int i = lane; __ballot(i < a.k); i += 64) {
      const float v = i < a.k ? a.isos[i] : 0.0f;
      j0 += __popcll(__ballot(i < a.k && v <= L));
      j1 += __popcll(__ballot(i < a.k && v < Hh));
    }
    if (!(L < Hh)) j1 = j0;
  }
  for (int jc = j0; jc < j1; jc += kApRound) {
    const int jn = min(kApRound, j1 - jc);
    // lane u holds isovalue u of the round and the wave's cells it passes through
    const float iso_u = lane < jn ? a.isos[jc + lane] : 0.0f;
    const int slot_u = lane < jn ? a.slot[jc + lane] : 0;
    uint32_t count_u = 0;
    for (int u = 0; u < jn; ++u) {
      const float iso = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(iso_u), u));
      const uint64_t m = __ballot(lo < iso) & __ballot(iso < hi);  // a corner below, one above
      if (m) count_u = lane == u ? (uint32_t)__popcll(m) : count_u;
    }
    if (lane < jn) s_wt[lane][w] = count_u;
    __syncthreads();
    if (w == 0) {
      uint32_t c[kApWaves] = {}, all = 0, sum;
      if (lane < jn)
#pragma unroll
        for (int q = 0; q < kApWaves; ++q) all += c[q] = s_wt[lane][q];
      uint32_t off = prefix32(all, sum);
      if (lane < jn) {
#pragma unroll
        for (int q = 0; q < kApWaves; ++q) {
          s_off[lane][q] = off;
          off += c[q];
        }
        if (all) atomicAdd(&a.counts[slot_u], all);
      }
      if (lane == 0) {
        s_base = sum ? atomicAdd(a.pool_count, (unsigned long long)sum) : 0ull;
        s_run = sum;
      }
    }
    __syncthreads();
    const int64_t base = (int64_t)s_base;
    if (s_run != 0) {  // block-uniform
      const uint32_t room = (uint32_t)min(max(a.cap - base, (int64_t)0), (int64_t)INT32_MAX);
      int32_t *const out = a.out + 3 * base;
      const uint32_t off_u = lane < jn ? s_off[lane][w] : 0u;
      for (uint64_t todo = __ballot(count_u != 0u); todo; todo &= todo - 1) {
        const int u = __ffsll((unsigned long long)todo) - 1;
        const float iso = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(iso_u), u));
        const uint64_t m = __ballot(lo < iso) & __ballot(iso < hi);
        const uint32_t pos = (uint32_t)__builtin_amdgcn_readlane((int)off_u, u) + lane_prefix(m);
        if (__builtin_amdgcn_inverse_ballot_w64(m) && pos < room) {
          *(int3 *)(out + 3u * pos) = make_int3(x, y, z);
          if (a.out_slot)
            a.out_slot[base + pos] = (uint32_t)__builtin_amdgcn_readlane(slot_u, u);
        }
      }
    }
    __syncthreads();  // s_base and s_run are written again by the next round
  }
}

}  // namespace

namespace iso {

int sort_vertices_lex(iso_ctx *ctx, float *d_xyz, int64_t n, int gx, int gy, int gz,
                      uint32_t *d_odd);

// Voxel approximation at k isovalues in one pass, pool output like mc_multi.
int approx_multi(iso_ctx *ctx, const float *d_img, int X, int Y, int Z, const float *d_isos_sorted,
                 const int *d_slot, int k, uint32_t *d_counts, int32_t *d_pool,
                 uint32_t *d_pool_slot, int64_t cap, int64_t *h_total) {
  *h_total = 0;
  ISO_TRY(fill_u32(ctx, d_counts, 0u, (size_t)k));
  if (X < 2 || Y < 2 || Z < 2 || k <= 0) return ISO_OK;
  if ((int64_t)(X - 1) * (Y - 1) * (Z - 1) > (int64_t)UINT32_MAX)
    return fail(ctx, ISO_ERR_UNSUPPORTED, "voxel approximation: more than 2^32-1 cells");
  void *ctr = nullptr, *pin = nullptr;
  ISO_TRY(ws_get(ctx, WS_MC_COUNTERS, 64, false, &ctr));
  ISO_TRY(fill_u32(ctx, ctr, 0u, 4));
  ApMultiArgs a;
  a.img = d_img;
  a.X = X;
  a.Y = Y;
  a.Z = Z;
  a.isos = d_isos_sorted;
  a.slot = d_slot;
  a.k = k;
  a.counts = d_counts;
  a.out = d_pool;
  a.out_slot = d_pool_slot;
  a.cap = d_pool ? cap : 0;
  a.pool_count = (unsigned long long *)ctr + 1;
  const int64_t blocks =
      (int64_t)((X - 1 + 3) / 4) * ((Y - 1 + 3) / 4) * ((Z - 1 + 15) / 16);
  hipLaunchKernelGGL(approx_multi_kernel, dim3((unsigned)blocks), dim3(kApBlock), 0, ctx->stream,
                     a);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  ISO_TRY(pinned_get(ctx, 16, &pin));
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(pin, ctr, 16, hipMemcpyDeviceToHost, ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  *h_total = (int64_t)((unsigned long long *)pin)[1];
  return ISO_OK;
}

// Marching cubes at k isovalues in one pass over the volume.  Every vertex
// goes to one pool (xyz, and its isovalue slot if d_pool_slot != null);
// counts/stats are device arrays indexed by slot (stats may be null: no cell
// statistics are then gathered); d_isos_sorted/d_slot give
// the ascending isovalues and their slots.  *h_total = vertices found, which
// may exceed cap (nothing past cap is written); h_counts (k words, may be
// null) receives the per-slot counts.  The vertex-writing pass is left
// running on the stream when this returns.  Synchronises the stream and
// retries when the grid-point hash set fills up.
int mc_multi(iso_ctx *ctx, const float *d_vol, int gx, int gy, int gz, uint32_t flags,
             const float *d_isos_sorted, const int *d_slot, int k, uint32_t *d_counts,
             unsigned long long *d_stats, float *d_pool, uint32_t *d_pool_slot, int64_t cap,
             int64_t *h_total, uint32_t *h_counts) {
  *h_total = 0;
  McArgs a;
  a.vol = d_vol;
  a.gx = gx;
  a.gy = gy;
  a.gz = gz;
  const bool compat = flags & ISO_COMPAT_MC;
  if (compat) {
    a.sx = 1;
    a.sy = gx;
    a.sz = (int64_t)gx * gy;
    a.ncx = gx;
    a.ncy = gy;
    a.ncz = gz;
    int64_t n = (int64_t)gx * gy * gz;
    int64_t bx = n / 128, by = 1;  // MarchingCube.cpp:599-608
    if (bx > 65535) { by = bx / 32768; bx = 32768; }
    a.ncls = std::min<int64_t>(128 * bx * by, n);
    a.zfast = 0;
  } else {
    a.sx = (int64_t)gy * gz;
    a.sy = gz;
    a.sz = 1;
    a.ncx = gx - 1;
    a.ncy = gy - 1;
    a.ncz = gz - 1;
    a.ncls = INT64_MAX;
    a.zfast = 1;
  }
  a.npx = a.ncx + 1;
  a.npy = a.ncy + 1;
  a.npz = a.ncz + 1;
  a.npoints = (int64_t)a.npx * a.npy * a.npz;
  // candidate vertex ids are 32-bit: point id * 5 + edge kind
  if (a.npoints > (int64_t)(UINT32_MAX / 5u))
    return fail(ctx, ISO_ERR_UNSUPPORTED,
                "marching cubes: %lld grid points, at most %u (32-bit candidate vertex ids)",
                (long long)a.npoints, UINT32_MAX / 5u);
  a.isos = d_isos_sorted;
  a.slot = d_slot;
  a.k = k;
  a.counts = d_counts;
  a.stats = d_stats;
  a.out = d_pool;
  a.out_slot = d_pool_slot;
  a.cap = d_pool ? cap : 0;
  memcpy(a.nverts, case_tables().nverts, 256);
  if (a.ncx <= 0 || a.ncy <= 0 || a.ncz <= 0 || k <= 0) {
    ISO_TRY(fill_u32(ctx, d_counts, 0u, (size_t)k));
    if (d_stats) ISO_TRY(fill_u32(ctx, d_stats, 0u, (size_t)4 * k));
    return ISO_OK;
  }
  const int64_t fast = a.zfast ? a.npz : a.npx, slow = a.zfast ? a.npx : a.npz;
  const int64_t blocks = ((fast + 15) / 16) * ((a.npy + 3) / 4) * ((slow + 3) / 4);
  void *blk = nullptr, *priv = nullptr, *tmp = nullptr;
  ISO_TRY(ws_get(ctx, WS_MC_BLOCKS, sizeof(uint32_t) * 2 * (size_t)(blocks + 1), false, &blk));
  // the count pass's vertices per (round, isovalue, wave) of each block, which
  // the emit pass starts each round from (every entry it reads is written)
  a.max_rounds = (k + kMcRound - 1) / kMcRound;
  void *wcb = nullptr;
  ISO_TRY(ws_get(ctx, WS_MC_WAVES,
                 sizeof(uint16_t) * (size_t)blocks * a.max_rounds * kMcRound * kMcWaves, false,
                 &wcb));
  a.wave_counts = (uint16_t *)wcb;
  ISO_TRY(ws_get(ctx, WS_MC_PRIV, (sizeof(uint32_t) + 2 * sizeof(unsigned long long)) * kMcPriv * (size_t)k,
                 false, &priv));
  ISO_TRY(ws_get(ctx, WS_SCAN_TMP, sizeof(uint32_t) * scan_tmp_words(blocks), false, &tmp));
  a.block_total = (uint32_t *)blk;
  a.block_base = (const uint32_t *)blk + (blocks + 1);
  a.stats_priv = (unsigned long long *)priv;
  a.counts_priv = (uint32_t *)(a.stats_priv + 2 * (size_t)kMcPriv * k);
  uint32_t log2cap = 16;
  for (int attempt = 0; attempt < 8; ++attempt, log2cap += 2) {
    const size_t slots = (size_t)1 << log2cap;
    void *tab = nullptr, *ctr = nullptr, *pin = nullptr;
    ISO_TRY(ws_get(ctx, WS_MC_CORNER_TABLE, slots * 12, false, &tab));  // keys, then owners
    ISO_TRY(ws_get(ctx, WS_MC_COUNTERS, 64, false, &ctr));
    // [overflow, vertex total, 64-bit vertex total, kMcOddVertices: of a sort to follow]
    ISO_TRY(fill3_u32(ctx, tab, 0xffffffffu, slots * 2, ctr, 0u, 5, priv, 0u, (size_t)kMcPriv * k * 5));
    a.corner_tab = (unsigned long long *)tab;
    a.corner_owner = (uint32_t *)(a.corner_tab + slots);
    a.corner_mask = (uint32_t)(slots - 1);
    a.overflow = (uint32_t *)ctr;
    // cell statistics only when the caller takes them
    if (d_stats)
      hipLaunchKernelGGL((mc_kernel<false, true>), dim3((unsigned)blocks), dim3(kMcBlock), 0,
                         ctx->stream, a);
    else
      hipLaunchKernelGGL((mc_kernel<false, false>), dim3((unsigned)blocks), dim3(kMcBlock), 0,
                         ctx->stream, a);
    ISO_HIP_CHECK(ctx, hipGetLastError());
    ISO_TRY(exclusive_scan_u32(ctx, a.block_total, (uint32_t *)a.block_base, blocks,
                               (uint32_t *)ctr + 1, (uint32_t *)tmp));
    hipLaunchKernelGGL(mc_reduce_kernel, dim3((unsigned)((k + 255) / 256)), dim3(256), 0,
                       ctx->stream, (const uint32_t *)a.counts_priv,
                       (const unsigned long long *)a.stats_priv, k, d_counts, d_stats,
                       (unsigned long long *)ctr + 1);
    // the counters, and the per-slot counts when the caller takes them (they
    // are final after the count pass), in one read-back
    ISO_TRY(pinned_get(ctx, 16 + (h_counts ? 4 * (size_t)k : 0), &pin));
    ISO_HIP_CHECK(ctx, hipMemcpyAsync(pin, ctr, 16, hipMemcpyDeviceToHost, ctx->stream));
    if (h_counts)
      ISO_HIP_CHECK(ctx, hipMemcpyAsync((char *)pin + 16, d_counts, 4 * (size_t)k,
                                        hipMemcpyDeviceToHost, ctx->stream));
    ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    if (((uint32_t *)pin)[0] != 0u) continue;  // grid-point table full: again, larger
    if (h_counts) memcpy(h_counts, (const char *)pin + 16, 4 * (size_t)k);
    *h_total = (int64_t)((uint32_t *)pin)[1];
    // the vertex offsets are a 32-bit scan: its total must be the exact one
    if ((unsigned long long)*h_total != ((unsigned long long *)pin)[1])
      return fail(ctx, ISO_ERR_UNSUPPORTED,
                  "marching cubes: %llu vertices over %d isovalues, at most %u per call",
                  ((unsigned long long *)pin)[1], k, UINT32_MAX);
    if (a.cap > 0 && *h_total <= a.cap && *h_total > 0)
      hipLaunchKernelGGL((mc_kernel<true, false>), dim3((unsigned)blocks), dim3(kMcBlock), 0,
                         ctx->stream,
                         a);
    ISO_HIP_CHECK(ctx, hipGetLastError());
    return ISO_OK;
  }
  return fail(ctx, ISO_ERR_OUT_OF_MEMORY, "marching cubes: grid-point vertex table overflow");
}

int approx_one(iso_ctx *ctx, const float *d_img, int X, int Y, int Z, float iso, int32_t *d_out,
               int64_t cap, int64_t *count) {
  *count = 0;
  if (X < 2 || Y < 2 || Z < 2) return ISO_OK;
  if ((int64_t)(X - 1) * (Y - 1) * (Z - 1) > (int64_t)UINT32_MAX)
    return fail(ctx, ISO_ERR_UNSUPPORTED, "voxel approximation: more than 2^32-1 cells");
  ApArgs a;
  a.img = d_img;
  a.X = X;
  a.Y = Y;
  a.Z = Z;
  a.ncells = (int64_t)(X - 1) * (Y - 1) * (Z - 1);
  a.iso = iso;
  a.out = d_out;
  a.cap = cap;
  const int64_t tiles = (a.ncells + kApTile - 1) / kApTile;
  void *cnt = nullptr, *tmp = nullptr;
  ISO_TRY(ws_get(ctx, WS_MC_KEYS_A, sizeof(uint32_t) * (tiles + 1), false, &cnt));
  ISO_TRY(ws_get(ctx, WS_SCAN_TMP, sizeof(uint32_t) * scan_tmp_words(tiles), false, &tmp));
  a.tile_counts = (uint32_t *)cnt;
  a.tile_offsets = (uint32_t *)cnt;
  hipLaunchKernelGGL(approx_count_kernel, dim3((unsigned)tiles), dim3(kApBlock), 0, ctx->stream, a);
  ISO_TRY(exclusive_scan_u32(ctx, (uint32_t *)cnt, (uint32_t *)cnt, tiles, (uint32_t *)cnt + tiles,
                             (uint32_t *)tmp));
  hipLaunchKernelGGL(approx_emit_kernel, dim3((unsigned)tiles), dim3(kApBlock), 0, ctx->stream, a);
  ISO_HIP_CHECK(ctx, hipGetLastError());
  uint32_t total = 0;
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(&total, (uint32_t *)cnt + tiles, 4, hipMemcpyDeviceToHost,
                                    ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  *count = total;
  return ISO_OK;
}

}  // namespace iso

extern "C" {

int iso_mc_extract(iso_ctx *ctx, const float *d_vol, int gx, int gy, int gz, float iso,
                   uint32_t flags, float *d_xyz, int64_t cap, int64_t *h_count,
                   iso_mc_stats *h_stats) {
  ISO_TRY(iso::enter(ctx));
  if (!d_vol || gx <= 0 || gy <= 0 || gz <= 0 || !h_count || cap < 0 || (cap > 0 && !d_xyz))
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_mc_extract: bad arguments");
  // one isovalue: small device block with [iso, slot, count, stats]
  struct Small {
    float iso;
    int slot;
    uint32_t count;
    uint32_t pad;
    unsigned long long stats[2];
  };
  void *dsm = nullptr, *pin = nullptr;
  ISO_TRY(iso::ws_get(ctx, WS_SMALL, sizeof(Small), false, &dsm));
  ISO_TRY(iso::pinned_get(ctx, 64, &pin));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  Small hs{};
  hs.iso = iso;
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(dsm, &hs, sizeof(Small), hipMemcpyHostToDevice, ctx->stream));
  Small *ds = (Small *)dsm;
  int64_t total = 0;
  ISO_TRY(iso::mc_multi(ctx, d_vol, gx, gy, gz, flags, &ds->iso, &ds->slot, 1, &ds->count,
                        ds->stats, d_xyz, nullptr, d_xyz ? cap : 0, &total, nullptr));
  ISO_HIP_CHECK(ctx, hipMemcpyAsync(&hs, dsm, sizeof(Small), hipMemcpyDeviceToHost, ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  *h_count = hs.count;
  if (h_stats) {
    h_stats->active_cells = (int64_t)hs.stats[0];
    h_stats->total_verts = (int64_t)hs.stats[1];
    h_stats->triangles = (int64_t)hs.stats[1] / 3;
    h_stats->unique_verts = hs.count;
  }
  if ((int64_t)hs.count > cap)
    return iso::fail(ctx, ISO_ERR_CAPACITY, "iso_mc_extract: %lld vertices, capacity %lld",
                     (long long)hs.count, (long long)cap);
  if ((flags & ISO_MC_SORTED) && hs.count > 1) {
    void *ctr = nullptr;
    ISO_TRY(iso::ws_get(ctx, WS_MC_COUNTERS, 64, false, &ctr));
    ISO_TRY(iso::sort_vertices_lex(ctx, d_xyz, hs.count, gx, gy, gz, (uint32_t *)ctr + kMcOddVertices));
  }
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  return ISO_OK;
}

int iso_approx_extract(iso_ctx *ctx, const float *d_img, int X, int Y, int Z, float iso,
                       int32_t *d_xyz, int64_t cap, int64_t *h_count) {
  ISO_TRY(iso::enter(ctx));
  if (!d_img || X <= 0 || Y <= 0 || Z <= 0 || !h_count || cap < 0 || (cap > 0 && !d_xyz))
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_approx_extract: bad arguments");
  int64_t n = 0;
  ISO_TRY(iso::approx_one(ctx, d_img, X, Y, Z, iso, d_xyz, cap, &n));
  *h_count = n;
  if (n > cap) return iso::fail(ctx, ISO_ERR_CAPACITY, "iso_approx_extract: %lld cells, capacity %lld", (long long)n, (long long)cap);
  return ISO_OK;
}

}  // extern "C"
