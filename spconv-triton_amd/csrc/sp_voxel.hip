// Point-cloud voxelisation (PointToVoxel) on gfx950.
//
// The reference (spconv_triton/pytorch/utils.py:72-163) quantises every point
// to a voxel, orders the voxels by the first point that falls in them
// ("first come, first served"), caps their number at max_num_voxels, and
// stores up to max_num_points_per_voxel points per voxel in arrival order,
// with torch.unique, scatter_reduce, argsort and cumsum.  Here:
//   1. insert: every in-range point's linear voxel key goes into an
//      open-addressing hash (sp_hash.h).  A slot keeps the smallest point index
//      (the voxel's first point) and counts its points; a point keeps its slot
//      and the count it met, a place of its own in the voxel's list;
//   2. number: a point is "first" when its slot holds its own index.  One scan
//      over the points, of first points and of their voxels' counts, numbers
//      the voxels in order of first occurrence (the FCFS ids) and says where
//      each one's list starts; the first point writes its voxel's clamped count
//      and coordinates (decoded from the key, ZYX order);
//   3. place: every point reads its voxel id (-1 past the cap) and enters
//      itself in its voxel's list, at the place it got from the insertion;
//   4. rank: a list is in no order, but a point's slot is the number of smaller
//      indices in it; points with slot < max_points_per_voxel are copied there.
// Step 4 reads a voxel's list once for each of its points, so where a voxel has
// too many points (p2v_rank_max) steps 3 and 4 are a stable radix sort of the points
// by voxel id instead (arrival order inside every voxel).
// The only host synchronisation is the read of the voxel count after step 2: it
// sizes the returned views (the reference reads it too: uniq.numel()), and the
// flag that comes with it chooses step 4.
#include "sp_common.h"
#include "sp_hash.h"
#include "sp_lookback.h"
#include "sp_sort.h"

namespace sp {

struct P2VGeom {
  int ndim;
  double vsize[4];
  double cmin[4];
  int64_t gsize[4];
};

// A voxel of the hash, in one 16-byte slot.  The insertion is bound by its atomics, which
// go past the XCD's L2 and queue up where points share a voxel.  So a plain read comes
// first, which spares the CAS where it shows the key (an old value costs one too many),
// and the points of a wave that share the voxel of its first one take one atomic for
// their count and one for the smallest index.  Whole calls against three atomics a
// point, us: 200k points of 134k voxels 116 and 115; 4M of 2.2M 1 586 and 1 394, of 20k
// 1 278 and 1 023; 1M of 64 821 and 1 065, of one 34 174 and 1 553.  (Reading the smallest
// index before its minimum as well: the few-voxel calls slower, 1 312 and 2 104.)
struct alignas(16) P2VSlot {
  uint64_t key;
  int32_t first;   // the smallest point index
  uint32_t count;  // its points; after the numbering its id
};
// Voxels of up to this many points are ranked by their lists (p2v_rank), which
// reads a voxel's list once per point, or about 3 maxpts of it where that is
// less; past about 16M reads the sort is the faster.  Whole calls, lists and
// sort, us: 200k points, 64 a voxel, all kept 128 and 140; 250 a voxel, 5 kept
// 134 and 152; 250, all kept 198 and 153; 1M points, 64 a voxel, all kept 459
// and 346; 250, 32 kept 422 and 318; 250, 8 kept 330 and 309.
static uint32_t p2v_rank_max(int64_t n, int maxpts) {
  const int64_t reads = (int64_t(1) << 24) / n;  // a point
  if (3 * int64_t(maxpts) <= reads) return 256u;
  return uint32_t(reads < 8 ? 8 : reads > 256 ? 256 : reads);
}
// counters in the workspace: scan chunks handed out, "a voxel has more than
// rank_max points", "the table is full"
enum { kMetaChunk = 0, kMetaLong = 16, kMetaOverflow = 17, kMetaWords = 64 };
struct P2VTable {
  P2VSlot* slots;
  uint64_t mask;
  uint32_t* overflow;

  // The slot of `key`, inserted when absent; -1 (and the overflow flag) when
  // the table is full.
  __device__ int64_t insert(uint64_t key) const {
    uint64_t s = mix64(key) & mask;
    for (uint64_t i = 0; i <= mask; ++i) {
      uint64_t have = __hip_atomic_load(&slots[s].key, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WAVEFRONT);
      if (have == kEmpty64)
        have = atomicCAS((unsigned long long*)&slots[s].key, (unsigned long long)kEmpty64,
                         (unsigned long long)key);
      if (have == kEmpty64 || have == key) return int64_t(s);
      s = (s + 1) & mask;
    }
    atomicExch(overflow, 1u);
    return -1;
  }
};

// The table, the counters and the voxels (n_vox floats), in one launch.
__global__ __launch_bounds__(256) void p2v_clear(uint4* __restrict__ slots, int64_t n_slots,
                                                 uint32_t* __restrict__ meta, int64_t n_meta,
                                                 float* __restrict__ voxels, int64_t n_vox) {
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  const int64_t t0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint4 none = make_uint4(0u, 0u, 0u, 0u);
  static_assert(kEmpty64 == ~uint64_t(0) && sizeof(P2VSlot) == 16, "an empty key is all ones");
  for (int64_t i = t0; i < n_slots; i += step) slots[i] = make_uint4(~0u, ~0u, 0x7fffffffu, 0u);
  for (int64_t i = t0; i < n_meta; i += step) meta[i] = 0u;
  const int64_t n4 = (reinterpret_cast<uintptr_t>(voxels) & 15) == 0 ? n_vox / 4 : 0;
  for (int64_t i = t0; i < n4; i += step) reinterpret_cast<uint4*>(voxels)[i] = none;
  for (int64_t i = 4 * n4 + t0; i < n_vox; i += step) voxels[i] = 0.f;
}

template <typename F>
__global__ __launch_bounds__(256) void p2v_insert(const F* __restrict__ pc, int64_t n,
                                                  int64_t cols, P2VGeom g, P2VTable t,
                                                  uint32_t rank_max, uint32_t* meta, int64_t* __restrict__ slot,
                                                  uint32_t* __restrict__ place) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  bool ok = i < n;
  int64_t lin = 0;
  for (int d = 0; i < n && d < g.ndim; ++d) {
    // (p - cmin) / vsize in the points' precision, as the reference computes
    // it with tensors of pc.dtype; the comparisons reject NaN as out of range
    const F q = floor((pc[i * cols + d] - F(g.cmin[d])) / F(g.vsize[d]));
    ok = ok && q >= F(0) && q < F(g.gsize[d]);
    lin = lin * g.gsize[d] + (ok ? int64_t(q) : 0);
  }
  const int64_t s = ok ? t.insert(uint64_t(lin)) : -1;
  const uint64_t in = __ballot(s >= 0);
  if (in != 0) {  // (wave-uniform)
    const int lane = int(threadIdx.x & 63), lead = __builtin_ctzll(in);
    const uint64_t same = __ballot(s == __shfl(s, lead, 64));  // (s >= 0 there)
    const bool shared = (same >> lane) & 1u;
    uint32_t before = 0;
    if (s >= 0 && (!shared || lane == lead)) {
      const uint32_t more = shared ? uint32_t(__popcll(same)) : 1u;
      before = atomicAdd(&t.slots[s].count, more);
      atomicMin(&t.slots[s].first, int32_t(i));  // (the lead lane's point is the first of its)
      if (before <= rank_max && rank_max - before < more) meta[kMetaLong] = 1u;
    }
    const uint32_t base = __shfl(before, lead, 64);
    if (shared) before = base + uint32_t(__popcll(same & lanemask_lt()));
    if (s >= 0) place[i] = before;
  }
  if (i < n) slot[i] = s;
}

// kNumThreads * kNumPer points a workgroup; the sums of the chunks before it by
// look-back, voxels in the low 31 bits of a state and points above them (both
// below 2^31).  A slot's count becomes the voxel's id: only its first point
// reads the count.  The last chunk's workgroup writes the totals to host
// memory: result[0] voxels, [1] whether one has more than rank_max points, [2]
// the table's overflow flag.
// Each chunk costs one atomic on the chunk counter, and these serialise: 391
// chunks of 512 points took 35 us (200k points, three atomics each), 196 of 1024
// with one each 15.3, 98 of 2048 19.0 (too few workgroups).
constexpr int kNumThreads = 512, kNumPer = 2, kNumChunk = kNumThreads * kNumPer;
__global__ __launch_bounds__(kNumThreads) void p2v_number(
    const int64_t* __restrict__ slot, int64_t n, int64_t chunks, P2VTable t, int64_t max_vox,
    int maxpts, P2VGeom g, uint32_t* __restrict__ counts,
    uint32_t* __restrict__ start, int32_t* __restrict__ npv, int32_t* __restrict__ indices,
    uint64_t* state, uint32_t* meta, uint64_t* __restrict__ result) {
  __shared__ uint32_t s_scan[2][kNumThreads / 64 + 1];
  __shared__ uint32_t s_chunk;
  __shared__ uint64_t s_base;
  if (threadIdx.x == 0) s_chunk = atomicAdd(&meta[kMetaChunk], 1u);
  __syncthreads();
  const int64_t chunk = s_chunk;
  if (chunk >= chunks) return;  // (a counter that was not cleared)
  const int64_t i0 = chunk * kNumChunk + int64_t(threadIdx.x) * kNumPer;
  int64_t sl[kNumPer];
  uint32_t c[kNumPer];
#pragma unroll
  for (int j = 0; j < kNumPer; ++j) sl[j] = i0 + j < n ? slot[i0 + j] : -1;
#pragma unroll
  for (int j = 0; j < kNumPer; ++j)
    c[j] = sl[j] >= 0 && t.slots[sl[j]].first == int32_t(i0 + j) ? t.slots[sl[j]].count : 0u;
  uint32_t nf = 0, np = 0;
#pragma unroll
  for (int j = 0; j < kNumPer; ++j) {
    nf += c[j] != 0u ? 1u : 0u;
    np += c[j];
  }
  uint32_t tot_f, tot_p;
  uint32_t vid = block_exclusive_scan<kNumThreads>(nf, s_scan[0], &tot_f);
  uint32_t at = block_exclusive_scan<kNumThreads>(np, s_scan[1], &tot_p);
  const uint64_t tot = uint64_t(tot_f) | (uint64_t(tot_p) << 31);
  if (threadIdx.x < 64) {
    const int lane = int(threadIdx.x);
    if (lane == 0)
      __hip_atomic_store(&state[chunk], (chunk == 0 ? kScanPrefix : kScanSum) | tot,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t base = scan_lookback(state, chunk, lane);
    if (lane == 0) {
      if (chunk != 0)
        __hip_atomic_store(&state[chunk], kScanPrefix | (base + tot), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      s_base = base;
      if (chunk == chunks - 1) {
        result[0] = (base + tot) & 0x7fffffffu;
        result[1] = meta[kMetaLong];
        result[2] = meta[kMetaOverflow];
      }
    }
  }
  __syncthreads();
  vid += uint32_t(s_base & 0x7fffffffu);
  at += uint32_t(s_base >> 31);
#pragma unroll
  for (int j = 0; j < kNumPer; ++j) {
    if (c[j] == 0u) continue;
    t.slots[sl[j]].count = vid;
    if (int64_t(vid) < max_vox) {
      counts[vid] = c[j];
      start[vid] = at;
      npv[vid] = int32_t(c[j] < uint32_t(maxpts) ? c[j] : uint32_t(maxpts));
      uint64_t key = t.slots[sl[j]].key;
      for (int d = g.ndim - 1; d >= 0; --d) {
        // (a 64-bit division takes several times a 32-bit one's instructions)
        const uint64_t size = uint64_t(g.gsize[d]);
        const uint64_t q = (key | size) >> 32 ? key / size : uint32_t(key) / uint32_t(size);
        indices[int64_t(vid) * g.ndim + (g.ndim - 1 - d)] = int32_t(key - q * size);  // ZYX
        key = q;
      }
    }
    ++vid;
    at += c[j];
  }
}

// Lists (list != null) or, for the sort, a key per point; pc_voxel_id either
// way.  place_vid[i], the point's place, becomes its voxel, or max_vox (dropped
// points sort last).
__global__ __launch_bounds__(256) void p2v_place(const int64_t* __restrict__ slot, int64_t n,
                                                 const P2VSlot* __restrict__ slots,
                                                 int64_t max_vox,
                                                 const uint32_t* __restrict__ start,
                                                 uint32_t* place_vid,
                                                 int64_t* __restrict__ pc_voxel_id,
                                                 uint32_t* __restrict__ list) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t s = slot[i];
  const uint32_t v = s >= 0 ? slots[s].count : 0u;
  const bool kept = s >= 0 && int64_t(v) < max_vox;
  pc_voxel_id[i] = kept ? int64_t(v) : -1;
  if (kept && list) list[start[v] + place_vid[i]] = uint32_t(i);
  place_vid[i] = kept ? v : uint32_t(max_vox);
}

// A point's slot: the smaller indices in its voxel's list, eight loads in
// flight, until there are maxpts of them.
template <typename F>
__global__ __launch_bounds__(256) void p2v_rank(const F* __restrict__ pc, int64_t n, int64_t cols,
                                                int nfeat, const uint32_t* __restrict__ vid,
                                                const uint32_t* __restrict__ counts,
                                                const uint32_t* __restrict__ start,
                                                const uint32_t* __restrict__ list,
                                                int64_t max_vox, int maxpts,
                                                float* __restrict__ voxels) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t v = vid[i];
  if (int64_t(v) >= max_vox) return;
  const uint32_t c = counts[v];
  const uint32_t* l = list + start[v];
  uint32_t r = 0;
  for (uint32_t j = 0; c > 1u && j < c && r < uint32_t(maxpts); j += 8) {
    uint32_t x[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) x[u] = l[j + u < c ? j + u : c - 1u];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) r += j + u < c && x[u] < uint32_t(i) ? 1u : 0u;
  }
  if (r >= uint32_t(maxpts)) return;
  float* dst = voxels + (int64_t(v) * maxpts + r) * nfeat;
  for (int f = 0; f < nfeat; ++f) dst[f] = float(pc[i * cols + f]);
}

template <typename F>
__global__ __launch_bounds__(256) void p2v_scatter(
    const F* __restrict__ pc, int64_t cols, int nfeat, const uint32_t* __restrict__ perm,
    const uint32_t* __restrict__ sort_key, const uint32_t* __restrict__ start, int64_t n,
    int64_t max_vox, int maxpts, float* __restrict__ voxels) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const uint32_t i = perm[p];
  const uint32_t v = sort_key[i];
  if (int64_t(v) >= max_vox) return;
  const int64_t slot = p - int64_t(start[v]);
  if (slot >= maxpts) return;
  float* dst = voxels + (int64_t(v) * maxpts + slot) * nfeat;
  for (int f = 0; f < nfeat; ++f) dst[f] = float(pc[int64_t(i) * cols + f]);
}

// Empty slots of every voxel get the mean over all max_points_per_voxel slots
// divided by the point count (reference utils.py:145-152), summed in slot order.
__global__ __launch_bounds__(256) void p2v_empty_mean(float* __restrict__ voxels,
                                                      const int32_t* __restrict__ npv,
                                                      int64_t nv, int maxpts, int nfeat) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= nv * nfeat) return;
  const int64_t v = t / nfeat;
  const int f = int(t % nfeat);
  float* base = voxels + v * maxpts * nfeat + f;
  float sum = 0.f;
  for (int s = 0; s < maxpts; ++s) sum += base[int64_t(s) * nfeat];
  const int cnt = npv[v];
  const float mean = sum / float(cnt > 1 ? cnt : 1);
  for (int s = cnt; s < maxpts; ++s) base[int64_t(s) * nfeat] = mean;
}

struct P2VWs {
  int64_t* slot;
  uint32_t* place;  // then vid
  uint32_t* counts;
  uint32_t* start;
  uint32_t* meta;
  uint64_t* state;
  P2VSlot* slots;
  void* sort_ws;  // the voxels' lists, or the sort's
  uint64_t cap;
  int64_t chunks;
};

template <class W>
static void p2v_layout(W& w, int64_t n, int64_t max_vox, P2VWs* out) {
  uint64_t cap = 1024;
  while (cap < uint64_t(n) * 2) cap <<= 1;
  const int64_t chunks = cdiv(n, kNumChunk);
  auto* slot = w.template take<int64_t>(size_t(n));
  auto* place = w.template take<uint32_t>(size_t(n));
  auto* counts = w.template take<uint32_t>(size_t(max_vox));
  auto* start = w.template take<uint32_t>(size_t(max_vox));
  auto* meta = w.template take<uint32_t>(kMetaWords + 2 * size_t(chunks));
  auto* slots = w.template take<P2VSlot>(size_t(cap));
  void* sws = w.template take<char>(sort_rows_ws_bytes(n));  // (at least 8 bytes a point)
  if (out) {
    out->slot = slot;
    out->place = place;
    out->counts = counts;
    out->start = start;
    out->meta = meta;
    out->state = reinterpret_cast<uint64_t*>(meta + kMetaWords);
    out->slots = slots;
    out->sort_ws = sws;
    out->cap = cap;
    out->chunks = chunks;
  }
}

// The size-only pass: WsSizer::take returns nothing, so the layout is walked
// with a cursor over a null base and only its final offset is used.
static size_t p2v_ws_bytes(int64_t n, int64_t max_vox) {
  WsCursor c(nullptr, ~size_t(0));
  p2v_layout(c, n, max_vox, nullptr);
  return c.off + 16;  // (the parts start at the workspace's first 16-byte boundary)
}

template <typename F>
static int p2v_run(const F* pc, int64_t n, int64_t cols, const P2VGeom& g, int nfeat,
                   int64_t max_vox, int maxpts, bool clear, bool empty_mean, float* voxels,
                   int32_t* indices, int32_t* npv, int64_t* pc_voxel_id, int64_t* n_voxels,
                   const P2VWs& w, hipStream_t s) {
  const unsigned blocks = unsigned(cdiv(n, 256));
  const P2VTable t{w.slots, w.cap - 1, w.meta + kMetaOverflow};
  PinnedCounts counts;
  int rc = counts.take();
  if (rc) return rc;
  const int64_t n_vox = clear ? max_vox * maxpts * nfeat : 0;
  const int64_t fb = cdiv(int64_t(w.cap) + n_vox / 4, 256);
  p2v_clear<<<unsigned(fb < 4096 ? fb : 4096), 256, 0, s>>>(
      reinterpret_cast<uint4*>(w.slots), int64_t(w.cap), w.meta, kMetaWords + 2 * w.chunks, voxels, n_vox);
  SP_LAUNCHED();
  p2v_insert<F><<<blocks, 256, 0, s>>>(pc, n, cols, g, t, p2v_rank_max(n, maxpts), w.meta, w.slot, w.place);
  SP_LAUNCHED();
  p2v_number<<<unsigned(w.chunks), kNumThreads, 0, s>>>(
      w.slot, n, w.chunks, t, max_vox, maxpts, g, w.counts, w.start, npv, indices,
      w.state, w.meta, counts.data());
  SP_LAUNCHED();
  SP_HIP(hipStreamSynchronize(s));
  const int64_t found = int64_t(counts.data()[0]);
  const int64_t nv = found < max_vox ? found : max_vox;
  if (counts.data()[2])
    return set_error(SP_ERR_HASH_FULL, "point2voxel: voxel hash overflowed");
  const bool lists = counts.data()[1] == 0;
  uint32_t* list = lists ? static_cast<uint32_t*>(w.sort_ws) : nullptr;
  p2v_place<<<blocks, 256, 0, s>>>(w.slot, n, w.slots, max_vox, w.start, w.place, pc_voxel_id,
                                   list);
  const uint32_t* vid = w.place;
  SP_LAUNCHED();
  if (lists) {
    p2v_rank<F><<<blocks, 256, 0, s>>>(pc, n, cols, nfeat, vid, w.counts, w.start, list, max_vox,
                                       maxpts, voxels);
    SP_LAUNCHED();
  } else {
    // stable sort of the points by voxel id (vid <= max_vox)
    int bits = 0;
    while ((uint64_t(1) << bits) <= uint64_t(max_vox)) ++bits;
    const uint32_t mask = bits >= 32 ? 0xFFFFFFFFu : ((1u << bits) - 1u);
    uint32_t* perm = nullptr;
    rc = sort_rows_by_words(vid, n, 1, bits, mask, &perm, w.sort_ws, s);
    if (rc) return rc;
    p2v_scatter<F><<<blocks, 256, 0, s>>>(pc, cols, nfeat, perm, vid, w.start, n, max_vox,
                                          maxpts, voxels);
    SP_LAUNCHED();
  }
  if (empty_mean && nv > 0) {
    const unsigned eblocks = unsigned(cdiv(nv * nfeat, 256));
    p2v_empty_mean<<<eblocks, 256, 0, s>>>(voxels, npv, nv, maxpts, nfeat);
    SP_LAUNCHED();
  }
  *n_voxels = nv;
  return SP_OK;
}

}  // namespace sp

using namespace sp;

extern "C" {

size_t sp_point2voxel_workspace_size(int64_t n_points, int64_t max_voxels) {
  if (n_points < 0 || max_voxels < 1) return 0;
  return p2v_ws_bytes(n_points > 0 ? n_points : 1, max_voxels);
}

int sp_point2voxel(const void* points, int32_t dtype, int64_t n_points, int64_t point_cols,
                   int32_t ndim, const double* vsize_xyz, const double* coors_min_xyz,
                   const int64_t* grid_size_xyz, int32_t num_point_features, int64_t max_voxels,
                   int32_t max_points_per_voxel, int32_t clear_voxels, int32_t empty_mean,
                   float* voxels, int32_t* indices, int32_t* num_per_voxel,
                   int64_t* pc_voxel_id, int64_t* num_voxels, void* ws, size_t ws_bytes,
                   void* stream) {
  SP_CHECK_ARG(ndim >= 1 && ndim <= 4, "point2voxel: ndim %d not in 1..4", ndim);
  SP_CHECK_ARG(dtype == SP_F32 || dtype == SP_F64, "point2voxel: points must be f32 or f64");
  SP_CHECK_ARG(n_points >= 0 && n_points < (int64_t(1) << 31), "point2voxel: bad point count");
  SP_CHECK_ARG(max_voxels >= 1 && max_voxels < (int64_t(1) << 31) && max_points_per_voxel >= 1,
               "point2voxel: bad capacities");
  SP_CHECK_ARG(num_point_features >= 1 && num_point_features <= point_cols && point_cols >= ndim,
               "point2voxel: %d point features of %lld columns", num_point_features,
               (long long)point_cols);
  SP_CHECK_ARG(vsize_xyz && coors_min_xyz && grid_size_xyz && num_voxels, "null pointer");
  *num_voxels = 0;
  P2VGeom g{};
  g.ndim = ndim;
  for (int d = 0; d < ndim; ++d) {
    SP_CHECK_ARG(grid_size_xyz[d] >= 1, "point2voxel: grid size %lld", (long long)grid_size_xyz[d]);
    g.vsize[d] = vsize_xyz[d];
    g.cmin[d] = coors_min_xyz[d];
    g.gsize[d] = grid_size_xyz[d];
  }
  hipStream_t s = as_stream(stream);
  if (n_points == 0) {
    if (clear_voxels)
      return launch_fill<float>(voxels, max_voxels * max_points_per_voxel * num_point_features,
                                0.f, s);
    return SP_OK;
  }
  SP_CHECK_ARG(points && voxels && indices && num_per_voxel && pc_voxel_id, "null pointer");
  const size_t need = p2v_ws_bytes(n_points, max_voxels);
  if (!ws || ws_bytes < need)
    return set_error(SP_ERR_WORKSPACE, "point2voxel: workspace %zu < %zu", ws_bytes, need);
  WsCursor c(reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(ws) + 15) & ~uintptr_t(15)),
             need - 16);
  P2VWs w;
  p2v_layout(c, n_points, max_voxels, &w);
  if (dtype == SP_F32)
    return p2v_run<float>(static_cast<const float*>(points), n_points, point_cols, g,
                          num_point_features, max_voxels, max_points_per_voxel, clear_voxels != 0,
                          empty_mean != 0, voxels, indices, num_per_voxel, pc_voxel_id, num_voxels,
                          w, s);
  return p2v_run<double>(static_cast<const double*>(points), n_points, point_cols, g,
                         num_point_features, max_voxels, max_points_per_voxel, clear_voxels != 0,
                         empty_mean != 0, voxels, indices, num_per_voxel, pc_voxel_id, num_voxels,
                         w, s);
}

}  // extern "C"
