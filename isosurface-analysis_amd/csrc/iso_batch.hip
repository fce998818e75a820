// Batched form over many volumes of uneven size: the ISMs of a whole batch.
//
// Per volume, extraction and distance fields run as in iso_ism_volume; the
// fields of every volume land in one buffer.  Then all unordered pairs of
// all ISMs go through persistent histogram+NMI launches: one or two workgroups
// per CU pull pair tasks (largest field first) from device queues until they
// are empty, so volumes from 48^3 to 256^3 share the machine without a launch,
// and its tail, per ISM.  One launch in the double form; in the reference's float
// order as many as the chains' inputs need room for, each with a launch that folds
// its chains (186,551 pairs at 128 bins: 32).
//
// Per-pair semantics are those of hist_nmi_kernel (JointHistogram.cu:24-162):
// exact integer joint counts privatised in LDS; NMI in the reference's float
// order with ISO_COMPAT_NMI32 (iso_nmi.hpp), else in double.
#include <algorithm>
#include <cstring>
#include <numeric>
#include <type_traits>
#include <vector>

#include "iso_bins.hpp"
#include "iso_df.hpp"
#include "iso_nmi.hpp"

namespace iso {
int mc_multi(iso_ctx *ctx, const float *d_vol, int gx, int gy, int gz, uint32_t flags,
             const float *d_isos_sorted, const int *d_slot, int k, uint32_t *d_counts,
             unsigned long long *d_stats, float *d_pool, uint32_t *d_pool_slot, int64_t cap,
             int64_t *h_total, uint32_t *h_counts);
int approx_multi(iso_ctx *ctx, const float *d_img, int X, int Y, int Z, const float *d_isos_sorted,
                 const int *d_slot, int k, uint32_t *d_counts, int32_t *d_pool,
                 uint32_t *d_pool_slot, int64_t cap, int64_t *h_total);
int field_interval(iso_ctx *ctx, const float *d_fields, int nfields, int64_t F, float *d_mins,
                   float *d_maxs);
}  // namespace iso

namespace {

struct BatchTask {
  int64_t fi, fj;  // element offsets of the two fields in the field buffer
  int64_t F;       // voxels per field
  int64_t processed;
  int mm_i, mm_j;  // the two fields' entries in the (mins, maxs) arrays
  int pad0, pad1;
  int map_i, map_j;  // entries (i,j) and (j,i) of the job's map
  int job, n;        // job index and its map size
};

struct BatchArgs {
  const float *fields;
  const float *mins, *maxs;  // per field of the batch (DistanceField::getInterval)
  const BatchTask *tasks;
  int ntasks;
  uint32_t *next;          // queue heads, cleared before each launch
  float *const *maps;      // per job: map (row-major n x n)
  uint32_t *ghist;         // per workgroup drain area (16-bit path), zero at rest
  int H;
  int nmi32;     // reference float-order NMI (ISO_COMPAT_NMI32)
  int hist_bytes;         // LDS histogram
  iso::ChainBufs chains;  // nmi32: the chains' inputs, per task
};

constexpr int kBBlock = iso::kHistBlock;

// The tasks come in tiles of 8 x 8 pairs of fields, and kTile tasks in a row go
// to one queue.  Workgroup b (XCD b % kQueues) takes from queue b % kQueues, so
// the pairs that run on an XCD at a time share 16 fields in its L2; when its
// queue is empty it goes on with the next one's.  31,054 pairs of 8 volumes, 128
// bins: 10.05 -> 9.1 ms against one queue in row order (tiles of 4 x 8: 9.5).
constexpr int kTileI = 8, kTileJ = 8, kTile = kTileI * kTileJ;
constexpr int kQueues = 8;
constexpr int kHeadStride = 8;  // words between two queue heads

// Everything a workgroup keeps in LDS, after the histogram.
template <bool PACK16>
struct BatchLds {
  iso::PairLds<PACK16> pair;
  double red[3][iso::kHistWaves];
  uint32_t prog[2];
  int task, flushed;
};

template <bool PACK16>
__global__ __launch_bounds__(kBBlock) __attribute__((amdgpu_waves_per_eu(PACK16 ? 4 : 8))) void hist_batch_kernel(BatchArgs a) {
  extern __shared__ uint4 s_dyn[];
  uint32_t *s_hist = reinterpret_cast<uint32_t *>(s_dyn);
  BatchLds<PACK16> &s = *reinterpret_cast<BatchLds<PACK16> *>(s_hist + a.H * iso::kRowWords<PACK16>);
  const int tid = threadIdx.x, H = a.H;
  const int words = H * iso::kRowWords<PACK16>;
  uint32_t *gh = a.ghist + (int64_t)blockIdx.x * H * H;
  int queue = blockIdx.x % kQueues, empty = 0;  // (lane 0's)
  while (true) {
    if (tid == 0) {
      int task;
      while (true) {
        const uint32_t i = atomicAdd(a.next + queue * kHeadStride, 1u);
        task = (int)min((i / kTile * kQueues + queue) * kTile + i % kTile, (uint32_t)a.ntasks);
        if (task < a.ntasks || ++empty == kQueues) break;
        queue = (queue + 1) % kQueues;
      }
      s.task = task;
      s.prog[0] = s.prog[1] = 0u;
      s.flushed = 0;
    }
    iso::clear_hist(s_hist, words);
    iso::clear_pair_lds(s.pair);
    __syncthreads();
    // wave-uniform (the LDS read is not known to be): the task's pointers
    // then live in scalar registers and the buffer resources built from them
    // need no per-lane waterfall
    const int ti = __builtin_amdgcn_readfirstlane(s.task);
    if (ti >= a.ntasks) break;
    const BatchTask t = a.tasks[ti];
    const float *f1 = a.fields + t.fi, *f2 = a.fields + t.fj;
    // the pair's bins (JointHistogram.cu:127-129): union range, H bins
    iso::PairBins<PACK16> bin;
    bin.init(fminf(a.mins[t.mm_i], a.mins[t.mm_j]), fmaxf(a.maxs[t.mm_i], a.maxs[t.mm_j]), H);
    for (int64_t b = 0; b < t.processed; b += iso::kMaxSlice) {  // (once)
      const int len = (int)min(iso::kMaxSlice, t.processed - b);
      auto accumulate = [&](auto sub) {
        constexpr bool SUB = decltype(sub)::value;
        if constexpr (PACK16)
          iso::accumulate16<SUB, 2>(bin, f1 + b, f2 + b, len, s_hist, s.prog, [&](int i, int j) {
            if (i >= H || j >= H) return;
            atomicAdd(&gh[i * H + j], 32768u);
            s.flushed = 1;
          });
        else
          iso::accumulate32<SUB, 4>(bin, f1 + b, f2 + b, len, s_hist);
      };
      if (__builtin_amdgcn_readfirstlane(bin.subtract)) accumulate(std::true_type());
      else accumulate(std::false_type());
      __syncthreads();
      if (tid == 0) s.prog[0] = s.prog[1] = 0u;
      __syncthreads();
    }
    uint32_t *src = nullptr;  // where the pair's counts are
    if (PACK16 && s.flushed) {
      src = gh;
      for (int w = tid; w < words; w += kBBlock) {
        const uint32_t v = s_hist[w];
        const int r = w / iso::kRowWords<PACK16>, c = 2 * (w % iso::kRowWords<PACK16>);
        if ((v & 0xffffu) && c < H) atomicAdd(&gh[r * H + c], v & 0xffffu);
        if ((v >> 16) && c + 1 < H) atomicAdd(&gh[r * H + c + 1], v >> 16);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __syncthreads();
    }
    // H made opaque here, so the tail's bin addresses are not hoisted out of
    // the task loop (they would stay live, and spill, across the histogram)
    int Hv = H;
    asm volatile("" : "+v"(Hv));
    if (a.nmi32) {
      // the chains of the reference's float order, folded by fold_batch_kernel
      const bool mirror = t.map_i != t.map_j;
      if (PACK16 && src)
        iso::emit_chains<PACK16, PACK16>(s_hist, a.hist_bytes, src, Hv, mirror, s.pair, a.chains, ti);
      else
        iso::emit_chains<PACK16, false>(s_hist, a.hist_bytes, nullptr, Hv, mirror, s.pair, a.chains,
                                        ti);
    } else {
      const double v = iso::nmi64_pair<PACK16>(s_hist, src, Hv, t.F, s.pair, s.red);
      if (tid == 0) {
        float *map = a.maps[t.job];
        map[(int64_t)t.map_i * t.n + t.map_j] = map[(int64_t)t.map_j * t.n + t.map_i] =
            (v != v) ? 0.0f : (float)v;
      }
    }
    __syncthreads();
  }
}

// The float-order NMI of every task of a hist_batch_kernel launch.
__global__ __launch_bounds__(64 * iso::kFoldWaves) void fold_batch_kernel(BatchArgs a) {
  __shared__ iso::FoldLds s_fold;
  const int64_t t0 = (int64_t)blockIdx.x * iso::kFoldPairs;
  iso::fold_chains(a.chains, a.H, t0, a.ntasks, [&](int64_t i) {
    const BatchTask t = a.tasks[i];
    float *map = a.maps[t.job];
    return iso::FoldOut{t.map_i != t.map_j, t.F, map + (int64_t)t.map_i * t.n + t.map_j,
                        map + (int64_t)t.map_j * t.n + t.map_i};
  }, s_fold);
}

}  // namespace

extern "C" {

int iso_ism_batch(iso_ctx *ctx, iso_ism_job *jobs, int njobs, int extractor, int ds, int H,
                  int df_method, uint32_t flags, iso_ism_stats *h_stats) {
  ISO_TRY(iso::enter(ctx));
  if (!jobs || njobs <= 0 || ds <= 0 || H < 1 || H > 256)
    return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_ism_batch: bad arguments");
  if (h_stats) memset(h_stats, 0, sizeof(*h_stats));
  // the stage events, destroyed on every return (early ones included)
  struct StageEvents {
    hipEvent_t e[3] = {nullptr, nullptr, nullptr};
    ~StageEvents() {
      for (auto &x : e)
        if (x) (void)hipEventDestroy(x);
    }
  } stage_events;
  hipEvent_t *ev = stage_events.e;
  for (int q = 0; q < 3; ++q) ISO_HIP_CHECK(ctx, hipEventCreate(&ev[q]));
  ISO_HIP_CHECK(ctx, hipEventRecord(ev[0], ctx->stream));
  // ---- per volume: extraction + distance fields into one field buffer
  std::vector<int64_t> fbase(njobs), F(njobs);
  int64_t ftotal = 0;
  for (int b = 0; b < njobs; ++b) {
    iso_ism_job &jb = jobs[b];
    if (!jb.d_vol || !jb.h_isos || !jb.d_map || !jb.h_ids || jb.k <= 0 || jb.X < ds ||
        jb.Y < ds || jb.Z < ds || jb.X < 2 || jb.Y < 2 || jb.Z < 2)
      return iso::fail(ctx, ISO_ERR_INVALID_ARG, "iso_ism_batch: bad job %d", b);
    F[b] = (int64_t)(jb.X / ds) * (jb.Y / ds) * (jb.Z / ds);
    fbase[b] = ftotal;
    ftotal += F[b] * jb.k;
  }
  void *fields = nullptr, *dmm = nullptr;
  ISO_TRY(iso::ws_get(ctx, WS_PIPE_E, sizeof(float) * (size_t)ftotal, false, &fields));
  int ktotal = 0;
  for (int b = 0; b < njobs; ++b) ktotal += jobs[b].k;
  // (mins, maxs) of every field of the batch, filled on the device
  ISO_TRY(iso::ws_get(ctx, WS_PIPE_D, sizeof(float) * 2 * (size_t)ktotal, false, &dmm));
  float *d_mins = (float *)dmm, *d_maxs = d_mins + ktotal;
  const bool mc = extractor == ISO_EXTRACT_MC;
  std::vector<BatchTask> tasks;
  std::vector<float *> maps(njobs);
  int64_t points = 0;
  int mmbase = 0;  // fields of the earlier jobs
  for (int b = 0; b < njobs; ++b) {
    iso_ism_job &jb = jobs[b];
    const int k = jb.k;
    std::vector<int> order(k);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return iso::iso_before(jb.h_isos[x], jb.h_isos[y]); });
    const size_t blk = 4 * (size_t)k * 2 + 4 * (size_t)k + 16 * (size_t)k;
    void *dblk = nullptr, *hblk = nullptr;
    ISO_TRY(iso::ws_get(ctx, WS_PIPE_A, blk + 1024, false, &dblk));
    ISO_TRY(iso::pinned_get(ctx, blk + 1024, &hblk));
    ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    float *h_iso = (float *)hblk;
    int *h_slot = (int *)(h_iso + k);
    for (int j = 0; j < k; ++j) {
      h_iso[j] = jb.h_isos[order[j]];
      h_slot[j] = order[j];
    }
    float *d_iso = (float *)dblk;
    int *d_slot = (int *)(d_iso + k);
    uint32_t *d_counts = (uint32_t *)(d_slot + k);
    ISO_HIP_CHECK(ctx, hipMemcpyAsync(dblk, hblk, 8 * (size_t)k, hipMemcpyHostToDevice, ctx->stream));
    int64_t total = 0;
    void *pool = nullptr, *pslot = nullptr;
    for (int attempt = 0; attempt < 2; ++attempt) {
      const int64_t cap = (int64_t)(ctx->ws[WS_PIPE_B].bytes / 12);
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_B, 12 * (size_t)std::max<int64_t>(cap, 1), false, &pool));
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_SLOTS, 4 * (size_t)std::max<int64_t>(cap, 1), false, &pslot));
      if (mc)
        ISO_TRY(iso::mc_multi(ctx, jb.d_vol, jb.X, jb.Y, jb.Z, flags, d_iso, d_slot, k, d_counts,
                              nullptr, (float *)pool, (uint32_t *)pslot, cap, &total, nullptr));
      else
        ISO_TRY(iso::approx_multi(ctx, jb.d_vol, jb.X, jb.Y, jb.Z, d_iso, d_slot, k, d_counts,
                                  (int32_t *)pool, (uint32_t *)pslot, cap, &total));
      if (total <= cap) break;
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_B, 12 * (size_t)total, false, &pool));
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_SLOTS, 4 * (size_t)total, false, &pslot));
    }
    std::vector<uint32_t> counts(k);
    ISO_HIP_CHECK(ctx, hipMemcpyAsync(counts.data(), d_counts, 4 * (size_t)k, hipMemcpyDeviceToHost,
                                      ctx->stream));
    ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    int m = 0;
    for (int j = 0; j < k; ++j)
      if (counts[j] > 0) jb.h_ids[m++] = j;
    jb.n_nonempty = m;
    maps[b] = jb.d_map;
    points += total;
    if (m == 0) continue;
    iso::SampleGrid g{jb.X, jb.Y, jb.Z, ds, jb.X / ds, jb.Y / ds, jb.Z / ds};
    float *fb = (float *)fields + fbase[b];
    ISO_TRY(iso::df_pool(ctx, pool, !mc, total, (const uint32_t *)pslot, k, counts.data(), g,
                         df_method, fb, false, /*coherent=*/true));
    // bin parameters come from the field intervals; the pair kernel reads
    // them on the device, so nothing is read back here
    ISO_TRY(iso::field_interval(ctx, fb, m, F[b], d_mins + mmbase, d_maxs + mmbase));
    int64_t processed = F[b];
    if ((flags & ISO_COMPAT_HIST_CHUNKS) && F[b] > 0 && F[b] % 1000000 == 0) processed -= 1000000;
    for (int i0 = 0; i0 < m; i0 += kTileI)
      for (int j0 = i0; j0 < m; j0 += kTileJ)
        for (int i = i0; i < std::min(m, i0 + kTileI); ++i)
          for (int j = std::max(i, j0); j < std::min(m, j0 + kTileJ); ++j) {
            BatchTask t;
            t.fi = fbase[b] + (int64_t)i * F[b];
            t.fj = fbase[b] + (int64_t)j * F[b];
            t.F = F[b];
            t.processed = processed;
            t.mm_i = mmbase + i;
            t.mm_j = mmbase + j;
            t.pad0 = t.pad1 = 0;
            t.map_i = i;
            t.map_j = j;
            t.job = b;
            t.n = m;
            tasks.push_back(t);
          }
    mmbase += m;
  }
  ISO_HIP_CHECK(ctx, hipEventRecord(ev[1], ctx->stream));
  // ---- all pairs of all ISMs: persistent launches, largest fields first
  std::stable_sort(tasks.begin(), tasks.end(),
                   [](const BatchTask &x, const BatchTask &y) { return x.F > y.F; });
  const int nt = (int)tasks.size();
  if (nt > 0) {
    const bool pack16 = H > 128;
    const int per_cu = pack16 ? 1 : 2;  // 1024-lane workgroups per CU (LDS)
    const int groups = std::min(nt, per_cu * ctx->cu_count);
    const bool nmi32 = (flags & ISO_COMPAT_NMI32) != 0;
    const size_t hist_bytes = sizeof(uint32_t) * (size_t)H * iso::row_words(H);
    const size_t lds = hist_bytes + (pack16 ? sizeof(BatchLds<true>) : sizeof(BatchLds<false>));
    // the LDS limit of the device's kernel, at the most bins' need: set to each
    // call's own, one thread could lower it between another's call and launch
    
    if (pack16)
      ISO_HIP_CHECK(ctx, hipFuncSetAttribute((const void *)hist_batch_kernel<true>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)(256 * 4 * iso::kRowWords<true> + sizeof(BatchLds<true>))));
    else
      ISO_HIP_CHECK(ctx, hipFuncSetAttribute((const void *)hist_batch_kernel<false>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)(128 * 4 * iso::kRowWords<false> + sizeof(BatchLds<false>))));
    BatchArgs ba;
    ba.fields = (const float *)fields;
    ba.mins = d_mins;
    ba.maxs = d_maxs;
    ba.H = H;
    ba.nmi32 = nmi32 ? 1 : 0;
    ba.hist_bytes = (int)hist_bytes;
    // tasks of a launch: what the memory for the chains' inputs holds (the tasks'
    // largest field comes first)
    const bool graph = (flags & ISO_BATCH_GRAPH) != 0;
    const int most = nmi32 ? iso::chain_tasks(ctx, H, tasks[0].F, nt, pack16 ? 2048 : 512) : nt;
    if (nmi32) ISO_TRY(iso::chain_get(ctx, most, H, tasks[0].F, ba.chains));
    auto launch = [&](const BatchTask *d_tasks) -> int {
      for (int i0 = 0; i0 < nt; i0 += most) {
        ba.tasks = d_tasks + i0;
        ba.ntasks = std::min(most, nt - i0);
        ISO_TRY(iso::fill_u32(ctx, ba.next, 0u, kQueues * kHeadStride));
        if (pack16)
          hipLaunchKernelGGL(hist_batch_kernel<true>, dim3(groups), dim3(kBBlock), lds, ctx->stream, ba);
        else
          hipLaunchKernelGGL(hist_batch_kernel<false>, dim3(groups), dim3(kBBlock), lds, ctx->stream, ba);
        if (nmi32)
          hipLaunchKernelGGL(fold_batch_kernel,
                             dim3((unsigned)((ba.ntasks + iso::kFoldPairs - 1) / iso::kFoldPairs)),
                             dim3(64 * iso::kFoldWaves), 0, ctx->stream, ba);
        ISO_HIP_CHECK(ctx, hipGetLastError());
      }
      return ISO_OK;
    };
    const size_t tbytes = sizeof(BatchTask) * (size_t)nt, mbytes = sizeof(float *) * (size_t)njobs;
    const size_t hbytes = sizeof(uint32_t) * (size_t)groups * H * H;
    if (graph) {
      // the graph owns one buffer: tasks | maps | queue heads | drain area; its
      // key is the layout: the tasks, the launch shape and the addresses of the
      // inputs and of the chains' inputs.  Those are the context's own, which
      // every launch fills anew: a workspace that has grown gets another address,
      // or at the same one holds what the graph needs, which has just been asked
      // for.
      uint64_t key = 1469598103934665603ull;
      auto mix = [&](const void *p, size_t n) {
        const unsigned char *c = (const unsigned char *)p;
        for (size_t i = 0; i < n; ++i) key = (key ^ c[i]) * 1099511628211ull;
      };
      mix(tasks.data(), tbytes);
      // every kernel argument the capture bakes in: d_maxs = d_mins + ktotal
      // moves with ktotal even where d_mins and the tasks stay the same
      const uint64_t shape[12] = {(uint64_t)H, (uint64_t)groups, (uint64_t)njobs,
                                 (uint64_t)(uintptr_t)fields, (uint64_t)(uintptr_t)d_mins,
                                 (uint64_t)(uintptr_t)d_maxs, (uint64_t)nt,
                                 (uint64_t)ba.nmi32, (uint64_t)lds, (uint64_t)most,
                                 (uint64_t)(uintptr_t)ba.chains.head,
                                 (uint64_t)(uintptr_t)ba.chains.logs};
      mix(shape, sizeof shape);
      iso_ctx::graph_entry *ge = nullptr;
      for (auto &e : ctx->graphs)
        if (e.key == key) ge = &e;
      const size_t o_maps = (tbytes + 255) & ~(size_t)255, o_head = o_maps + ((mbytes + 255) & ~(size_t)255);
      const size_t o_hist = o_head + 256, need = o_hist + hbytes;
      if (!ge) {
        if (ctx->graphs.size() >= 8) {  // keep a few layouts: drop the oldest
          ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
          auto &old = ctx->graphs.front();
          if (old.exec) (void)hipGraphExecDestroy(old.exec);
          if (old.buf) (void)hipFree(old.buf);
          ctx->graphs.erase(ctx->graphs.begin());
        }
        iso_ctx::graph_entry e;
        e.key = key;
        e.bytes = need;
        ISO_HIP_CHECK(ctx, hipMalloc(&e.buf, need));
        char *gb = (char *)e.buf;
        ISO_HIP_CHECK(ctx, hipMemcpyAsync(gb, tasks.data(), tbytes, hipMemcpyHostToDevice, ctx->stream));
        ISO_TRY(iso::fill_u32(ctx, gb + o_hist, 0u, hbytes / 4));  // drain area: zero at rest
        ba.maps = (float *const *)(gb + o_maps);
        ba.next = (uint32_t *)(gb + o_head);
        ba.ghist = (uint32_t *)(gb + o_hist);
        hipGraph_t captured = nullptr;
        ISO_HIP_CHECK(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        const int rc = launch((const BatchTask *)gb);
        const hipError_t ce = hipStreamEndCapture(ctx->stream, &captured);
        if (rc != ISO_OK) {
          if (captured) (void)hipGraphDestroy(captured);
          (void)hipFree(e.buf);
          return rc;
        }
        ISO_HIP_CHECK(ctx, ce);
        const hipError_t ie = hipGraphInstantiate(&e.exec, captured, nullptr, nullptr, 0);
        (void)hipGraphDestroy(captured);
        if (ie != hipSuccess) {
          (void)hipFree(e.buf);
          ISO_HIP_CHECK(ctx, ie);
        }
        ctx->graphs.push_back(e);
        ge = &ctx->graphs.back();
      } else {
        ++ge->replays;
      }
      // the maps may be new buffers each call: refresh their addresses
      ISO_HIP_CHECK(ctx, hipMemcpyAsync((char *)ge->buf + o_maps, maps.data(), mbytes,
                                        hipMemcpyHostToDevice, ctx->stream));
      ISO_HIP_CHECK(ctx, hipGraphLaunch(ge->exec, ctx->stream));
      if (h_stats) h_stats->graph_replays = ge->replays;
    } else {
      void *dt = nullptr, *dq = nullptr, *dmaps = nullptr, *gh = nullptr;
      ISO_TRY(iso::ws_get(ctx, WS_HIST_TASKS, tbytes, false, &dt));
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_G, 256, false, &dq));
      ISO_TRY(iso::ws_get(ctx, WS_PIPE_F, mbytes, false, &dmaps));
      ISO_TRY(iso::ws_get(ctx, WS_HIST_GLOBAL, hbytes, true, &gh));
      ISO_HIP_CHECK(ctx, hipMemcpyAsync(dt, tasks.data(), tbytes, hipMemcpyHostToDevice,
                                        ctx->stream));
      ISO_HIP_CHECK(ctx, hipMemcpyAsync(dmaps, maps.data(), mbytes, hipMemcpyHostToDevice,
                                        ctx->stream));
      ba.next = (uint32_t *)dq;
      ba.maps = (float *const *)dmaps;
      ba.ghist = (uint32_t *)gh;
      ISO_TRY(launch((const BatchTask *)dt));
    }
  }
  ISO_HIP_CHECK(ctx, hipEventRecord(ev[2], ctx->stream));
  ISO_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
  if (h_stats) {
    float t01 = 0, t12 = 0;
    (void)hipEventElapsedTime(&t01, ev[0], ev[1]);
    (void)hipEventElapsedTime(&t12, ev[1], ev[2]);
    int ne = 0;
    for (int b = 0; b < njobs; ++b) ne += jobs[b].n_nonempty;
    h_stats->n_nonempty = ne;
    h_stats->total_points = points;
    h_stats->ms_df = t01;  // extraction + fields of all volumes
    h_stats->ms_hist = t12;
  }
  return ISO_OK;
}

}  // extern "C"
