// Device-side planning of one attention step: the extend work list of
// tf_attn_plan_extend and the decode item list of tf_attn_plan_decode_items,
// built on the GPU from the device extend_lens, so a step needs no host loop
// and no host->device copy and can be captured in a HIP graph.
//
// The host-side bookkeeping this replaces is the reference's per-step index
// work around the extend branch (qwen3_8/full_attention.py:250-265: q_start
// prefix sums and the per-request row split) and the caller's per-step host
// metadata (engine/model_runner.py:108-188).  The lists are identical to the
// host planners' (same order: largest extend first, later row tiles first, kv
// heads inner) and are padded to capacities the host knows without reading
// device memory:
//   work:  kv_heads * (ceil(T * G / 256) + B) entries, padding {0,0,0,0,0,...}
//          (ext 0: the extend kernels skip it);
//   decode items: B entries, padding -1 (the decode kernels skip it).
#include "tf_common.h"
#include "tf_internal.h"

namespace tfa {
namespace {

constexpr int kPlanMaxBatch = 4096;
constexpr int kPlanThreads = 1024;
constexpr int kPlanPer = kPlanMaxBatch / kPlanThreads;   // requests per thread

struct PlanArgs {
  const int64_t* ext;
  int32_t batch, hkv, group, dec_to_dec;
  int32_t* work;
  int32_t work_cap;
  int32_t* dec_items;
  int32_t* dec_rows;
  int32_t dec_cap;
  int32_t* status;
};

struct PlanSmem {
  int32_t ext[kPlanMaxBatch];        // extend length per request (0 if absent)
  int32_t qs[kPlanMaxBatch];         // first q row of each request
  int32_t order[kPlanMaxBatch];      // extend requests, largest first
  int32_t off[kPlanMaxBatch + 1];    // first work entry of the request at rank r
  int64_t wsum[kPlanThreads / kWave];
};

// Exclusive block-wide prefix sum of one value per thread; returns the prefix
// and sets total.  All threads must call it.
__device__ int64_t block_scan(int64_t v, int64_t* wsum, int64_t& total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  int64_t x = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int64_t y = __shfl_up(x, d, kWave);
    if (lane >= d) x += y;
  }
  __syncthreads();
  if (lane == kWave - 1) wsum[w] = x;
  __syncthreads();
  int64_t before = 0;
  total = 0;
  for (int k = 0; k < kPlanThreads / kWave; ++k) {
    if (k < w) before += wsum[k];
    total += wsum[k];
  }
  return before + x - v;
}

__global__ void __launch_bounds__(kPlanThreads) plan_kernel(PlanArgs a) {
  __shared__ PlanSmem sm;
  const int tid = threadIdx.x;
  const int G = a.group;

  // Requests tid * kPlanPer + k: lengths, q_start, decode / extend roles.
  int32_t e[kPlanPer];
  bool bad = false;
  int64_t tok = 0;
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    const int b = tid * kPlanPer + k;
    int64_t x = b < a.batch ? a.ext[b] : 0;
    if (b < a.batch && (x < 1 || x > INT32_MAX)) {
      bad = true;
      x = 0;
    }
    e[k] = (int32_t)x;
    tok += x;
  }
  int64_t total_tok;
  int64_t q0 = block_scan(tok, sm.wsum, total_tok);
  int64_t q_start[kPlanPer];
  int ndec = 0, next = 0;
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    q_start[k] = q0;
    sm.qs[tid * kPlanPer + k] = (int32_t)min<int64_t>(q0, INT32_MAX);
    q0 += e[k];
    const bool dec = e[k] == 1 && a.dec_to_dec;
    const bool ext = e[k] >= 1 && !dec;
    sm.ext[tid * kPlanPer + k] = ext ? e[k] : 0;
    ndec += dec;
    next += ext;
  }

  // Decode items in request order.
  int64_t n_dec64, n_ext64;
  int64_t d0 = block_scan(ndec, sm.wsum, n_dec64);
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    if (e[k] == 1 && a.dec_to_dec) {
      if (d0 < a.dec_cap) {
        a.dec_items[d0] = tid * kPlanPer + k;
        a.dec_rows[d0] = (int32_t)q_start[k];
      }
      ++d0;
    }
  }
  (void)block_scan(next, sm.wsum, n_ext64);
  __syncthreads();   // sm.ext complete

  // Rank of each extend request: larger extend first, then request order.
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    const int b = tid * kPlanPer + k;
    const int x = sm.ext[b];
    if (x == 0) continue;
    int rank = 0;
    for (int c = 0; c < a.batch; ++c) {
      const int y = sm.ext[c];
      rank += (y > x) || (y == x && y != 0 && c < b);
    }
    sm.order[rank] = b;
  }
  __syncthreads();

  // Work entries per rank: kv_heads x row tiles of the request.
  int64_t cnt = 0;
  int32_t n_r[kPlanPer];
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    const int r = tid * kPlanPer + k;
    n_r[k] = 0;
    if (r < n_ext64) {
      const int64_t rows = (int64_t)sm.ext[sm.order[r]] * G;
      n_r[k] = (int32_t)(a.hkv * ((rows + kExtendItemRows - 1) / kExtendItemRows));
    }
    cnt += n_r[k];
  }
  int64_t n_work64;
  int64_t w0 = block_scan(cnt, sm.wsum, n_work64);
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    sm.off[tid * kPlanPer + k] = (int32_t)min<int64_t>(w0, INT32_MAX);
    w0 += n_r[k];
  }
  if (tid == 0) sm.off[kPlanMaxBatch] = (int32_t)min<int64_t>(n_work64, INT32_MAX);
  __syncthreads();

  // Entries, one thread each: rank by binary search over the offsets, then
  // (tile from the last, kv head inner) within the request.  Entries past the
  // real ones are padding (ext 0).
  const int n_work = (int)min<int64_t>(n_work64, a.work_cap);
  for (int idx = tid; idx < a.work_cap; idx += kPlanThreads) {
    int32_t* wk = a.work + 8 * (int64_t)idx;
    int32_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (idx < n_work) {
      int lo = 0, hi = (int)n_ext64 - 1;   // last rank with off <= idx
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sm.off[mid] <= idx) lo = mid; else hi = mid - 1;
      }
      const int b = sm.order[lo];
      const int x = sm.ext[b];
      const int tiles = (int)(((int64_t)x * G + kExtendItemRows - 1) / kExtendItemRows);
      const int j = idx - sm.off[lo];
      const int t = tiles - 1 - j / a.hkv;
      v[0] = b;
      v[1] = j % a.hkv;
      v[2] = t * kExtendItemRows;
      v[3] = sm.qs[b];
      v[4] = x;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) wk[q] = v[q];
  }
  for (int i = (int)min<int64_t>(n_dec64, a.dec_cap) + tid; i < a.dec_cap; i += kPlanThreads) {
    a.dec_items[i] = -1;
    a.dec_rows[i] = 0;
  }
  const bool any_bad = __syncthreads_or(bad);
  if (tid == 0) {
    a.status[0] = (int32_t)min<int64_t>(n_work64, INT32_MAX);
    a.status[1] = (int32_t)n_dec64;
    a.status[2] = (any_bad ? 2 : 0) | (n_work64 > a.work_cap || n_dec64 > a.dec_cap ? 1 : 0);
  }
}

// ---------------------------------------------------------------------------
// Which kernel a request's rows take: the row blocks of the streaming kernel
// (tf_attn_rows) and the work entries left to the extend kernel, from the work
// list and the decode items of a step (host- or device-planned, padding
// included).  Requests of at most max_rows rows (ext * G) go to the streaming
// kernel, in blocks of a unit's rows.
struct BlockArgs {
  const int32_t* work;
  int32_t n_work;
  const int32_t* dec_items;
  const int32_t* dec_rows;
  int32_t n_dec;
  int32_t group, unit_rows;
  int64_t max_rows;       // entries of requests with at most this many rows go to blocks
  RowItem* blocks;
  int32_t n_blocks;
  int32_t* pieces;
  int32_t n_pieces;
  int32_t* merges;        // NULL: entries are not split
  int32_t n_merges;
  const int64_t* seq_lens;
  int32_t seq_override;
  int64_t rtt_cols;
  int32_t key_bytes;      // K and V of one token
  int32_t cus;
};

// Key split of the extend kernel's entries.  A workgroup of that kernel fills a
// CU and walks its entry's keys in order, so with fewer entries than CUs the
// longest entry's keys set the time.  The entries are then cut into pieces of
// about equal key counts, at most one per CU, whose fp32 partials a merge
// launch combines.  In tiles of 32 keys (about 1.5 us each): an entry costs its
// tiles + 15 (Q, first slots, output), a piece its tiles + 24 (it also writes
// 256 KB of partials), the merge 3 + 0.047 per piece.  The shortest piece
// length that gives no more pieces than CUs is taken when it beats the whole
// entries by 8 %; short contexts (below about 900 keys) never do.  The step's
// streaming rows (decodes, short extends) run beside whole entries, on the CUs
// these leave, but after pieces that take every CU: their keys' time at 6 TB/s
// counts in full against the split (86 decodes on 100 to 4k keys beside 2 prompts
// of 260 tokens on 1k to 3k: 175 us whole, 203 split).  Measured
// (24 / 4 heads): 3 requests of 37 to 211 new tokens on 1.5k to 6k keys, 36
// entries of up to 180 tiles: 252 us whole, 48 + 14 (merge) in 252 pieces.  One
// of 2000 tokens on 3000, 188 entries of 95 to 156 tiles, stays whole (the plan
// would save a tenth of the kernel and pay it back in the merge).
constexpr int kSplitMax = 512;      // entries a split is considered for (LDS)
constexpr int kMinPiece = 12;       // tiles
constexpr float kEntryCost = 15.f, kPieceCost = 24.f, kMergeCost = 3.f, kMergePiece = 0.047f;

struct SplitSmem {
  int32_t src[kSplitMax];     // index of the kept entry in the work list
  int32_t tiles[kSplitMax];
  int32_t piece;              // tiles per piece (0: no split)
};

__device__ __forceinline__ int64_t context_len(const BlockArgs& a, int b) {
  const int64_t len = a.seq_override > 0 ? (int64_t)a.seq_override : a.seq_lens[b];
  return min(max(len, (int64_t)0), a.rtt_cols);
}

// Tiles of 32 keys that the entry's rows see.
__device__ __forceinline__ int entry_tiles(const BlockArgs& a, const int32_t* wk) {
  const int64_t len = context_len(a, wk[0]);
  const int64_t last = min<int64_t>((int64_t)wk[2] + kExtendItemRows, (int64_t)wk[4] * a.group) - 1;
  const int64_t kend = min(len, len - wk[4] + last / a.group + 1);
  return kend > 0 ? (int)((kend + 31) / 32) : 0;
}

// Tiles per piece for n entries, by wave 0 (every lane gets it; 0: no split).
// rows: the streaming rows' time, in tiles.
__device__ int piece_tiles(const SplitSmem& sm, int n, int cus, float rows) {
  const int lane = threadIdx.x & (kWave - 1);
  auto wave_sum = [&](int v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, kWave);
    return v;
  };
  int sum = 0, mx = 0;
  for (int i = lane; i < n; i += kWave) {
    sum += sm.tiles[i];
    mx = max(mx, sm.tiles[i]);
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) mx = max(mx, __shfl_xor(mx, d, kWave));
  if (n > cus || mx < 2 * kMinPiece) return 0;
  auto pieces = [&](int len) {
    int k = 0;
    for (int i = lane; i < n; i += kWave) k += (sm.tiles[i] + len - 1) / len;
    return wave_sum(k);
  };
  int lo = kMinPiece, hi = mx;   // pieces(mx) <= n <= cus
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pieces(mid) <= cus) hi = mid; else lo = mid + 1;
  }
  const float split = (float)hi + kPieceCost + kMergeCost + kMergePiece * (float)pieces(hi) + rows;
  return split < 0.92f * fmaxf((float)mx + kEntryCost, rows) ? hi : 0;
}

__global__ void __launch_bounds__(kPlanThreads) blocks_kernel(BlockArgs a) {
  __shared__ int64_t wsum[kPlanThreads / kWave];
  __shared__ SplitSmem sm;
  const int tid = threadIdx.x;
  const int R = a.unit_rows, G = a.group;
  int64_t at = 0;   // blocks so far
  int64_t keys = 0;   // of the streaming rows
  auto emit = [&](int n, int64_t i0, const RowItem& first) {
    for (int k = 0; k < n; ++k)
      if (i0 + k < a.n_blocks)
        a.blocks[i0 + k] = RowItem{first.b, first.qrow, first.ext, first.row0 + k * R};
  };
  for (int base = 0; base < a.n_dec; base += kPlanThreads) {
    const int i = base + tid;
    RowItem it{-1, 0, 1, 0};
    if (i < a.n_dec) {
      it.b = a.dec_items[i];
      it.qrow = a.dec_rows[i];
    }
    const int n = it.b < 0 ? 0 : (G + R - 1) / R;
    int64_t total;
    const int64_t before = block_scan(n, wsum, total);
    emit(n, at + before, it);
    at += total;
    if (a.merges) {
      (void)block_scan(it.b < 0 ? 0 : context_len(a, it.b), wsum, total);
      keys += total;
    }
  }
  int64_t kept = 0;   // pieces so far
  for (int base = 0; base < a.n_work; base += kPlanThreads) {
    const int i = base + tid;
    int32_t wk[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (i < a.n_work) {
#pragma unroll
      for (int q = 0; q < 8; ++q) wk[q] = a.work[8 * (int64_t)i + q];
    }
    const int64_t rows = (int64_t)wk[4] * G;
    const bool to_blocks = rows > 0 && (rows <= a.max_rows);
    const RowItem it{wk[0], wk[3], wk[4], wk[2]};
    const int n = to_blocks && wk[1] == 0
                      ? (int)((min<int64_t>(kExtendItemRows, rows - wk[2]) + R - 1) / R) : 0;
    int64_t total;
    const int64_t before = block_scan(n, wsum, total);
    emit(n, at + before, it);
    at += total;
    if (a.merges) {
      const bool first = n > 0 && wk[2] == 0;
      (void)block_scan(first ? context_len(a, wk[0]) : 0, wsum, total);
      keys += total;
    }
    const bool keep = rows > 0 && !to_blocks;
    int64_t n_keep;
    const int64_t k0 = kept + block_scan(keep ? 1 : 0, wsum, n_keep);
    if (keep && k0 < a.n_pieces) {
#pragma unroll
      for (int q = 0; q < 8; ++q) a.pieces[8 * k0 + q] = wk[q];
    }
    if (keep && a.merges && k0 < kSplitMax) {
      sm.src[k0] = i;
      sm.tiles[k0] = entry_tiles(a, wk);
    }
    kept += n_keep;
  }
  int64_t n_merge = 0;
  if (a.merges && kept <= kSplitMax) {
    __syncthreads();
    if (tid < kWave) {
      // a tile takes about 1.5 us, 9 MB at 6 TB/s
      const int len = piece_tiles(sm, (int)kept, a.cus, (float)keys * (float)a.key_bytes / 9e6f);
      if (tid == 0) sm.piece = len;
    }
    __syncthreads();
    const int len = sm.piece;
    if (len > 0) {   // kSplitMax <= kPlanThreads: one entry per thread
      const int t = tid < kept ? sm.tiles[tid] : 0;
      const int n = tid < kept ? max(1, (t + len - 1) / len) : 0;
      int64_t total, slots;
      const int64_t p0 = block_scan(n, wsum, total);
      const int64_t s0 = block_scan(n > 1 ? n : 0, wsum, slots);
      const int64_t m0 = block_scan(n > 1 ? 1 : 0, wsum, n_merge);
      // (more merges than the caller has room for: the entries stay whole)
      if (n_merge <= a.n_merges && tid < kept) {
        int32_t wk[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) wk[q] = a.work[8 * (int64_t)sm.src[tid] + q];
        for (int k = 0; k < n && p0 + k < a.n_pieces; ++k) {
          int32_t* pc = a.pieces + 8 * (p0 + k);
#pragma unroll
          for (int q = 0; q < 5; ++q) pc[q] = wk[q];
          pc[5] = n > 1 ? (int)((int64_t)t * k / n) : 0;
          pc[6] = n > 1 ? (int)((int64_t)t * (k + 1) / n) : 0;
          pc[7] = n > 1 ? (int32_t)(s0 + k + 1) : 0;
        }
        if (n > 1) {
          int32_t* mg = a.merges + 8 * m0;
#pragma unroll
          for (int q = 0; q < 5; ++q) mg[q] = wk[q];
          mg[5] = (int32_t)s0;
          mg[6] = n;
          mg[7] = 0;
        }
      }
      if (n_merge <= a.n_merges)
        kept = total;
      else
        n_merge = 0;
    }
  }
  if (a.merges)
    for (int64_t i = 8 * n_merge + tid; i < 8LL * a.n_merges; i += kPlanThreads) a.merges[i] = 0;
  for (int64_t i = at + tid; i < a.n_blocks; i += kPlanThreads)
    a.blocks[i] = RowItem{-1, 0, 1, 0};
  for (int64_t i = 8 * kept + tid; i < 8LL * a.n_pieces; i += kPlanThreads) a.pieces[i] = 0;
}

// ---------------------------------------------------------------------------
// req_to_token sync: the per-step incremental update of the resident device
// req_to_token table (engine/model_runner.py:147-167) as one kernel.  Request
// b of the batch owns two runs of flat elements, its rewritten prefix positions
// [patch_from, prefix) read from patch_vals, then its new positions
// [prefix, seq) read from out_cache_loc; every workgroup scans the run lengths
// of the whole batch into LDS and then takes flat elements in a grid-stride
// loop, finding each element's request by binary search.
constexpr int kSyncMaxBatch = kPlanMaxBatch;

struct SyncArgs {
  int64_t* table;
  int64_t rows, stride, cols;
  const int64_t* rpi;
  const int64_t* prefix;
  const int64_t* seq;
  const int64_t* loc;
  int64_t loc_len;
  const int64_t* pfrom;   // NULL: no rewritten prefixes
  const int64_t* poff;
  const int64_t* pvals;
  int64_t pvals_len;
  int32_t batch;
};

struct SyncSmem {
  int64_t flat[kSyncMaxBatch + 1];   // first flat element of request b
  int64_t loc[kSyncMaxBatch];        // first out_cache_loc entry of request b
  int64_t wsum[kPlanThreads / kWave];
};

// What request b writes.  A request whose row or range is outside the table
// (row outside [0, rows), not 0 <= prefix <= seq <= cols) writes nothing and
// takes no out_cache_loc entries; a patch run outside [0, prefix) or past the
// end of patch_vals is dropped.
struct SyncReq {
  int64_t row, prefix, pfrom, poff, n_patch, n_new;
};

__device__ __forceinline__ SyncReq sync_req(const SyncArgs& a, int b) {
  SyncReq q{0, 0, 0, 0, 0, 0};
  const int64_t r = a.rpi[b], p = a.prefix[b], s = a.seq[b];
  if (r < 0 || r >= a.rows || p < 0 || p > s || s > a.cols) return q;
  q.row = r;
  q.prefix = p;
  q.n_new = s - p;
  if (a.pfrom) {
    const int64_t f = a.pfrom[b], o = a.poff[b];
    if (f >= 0 && f < p && o >= 0 && o <= a.pvals_len - (p - f)) {
      q.pfrom = f;
      q.poff = o;
      q.n_patch = p - f;
    }
  }
  return q;
}

__global__ void __launch_bounds__(kPlanThreads) rtt_sync_kernel(SyncArgs a) {
  __shared__ SyncSmem sm;
  const int tid = threadIdx.x;
  int64_t n_el[kPlanPer], n_loc[kPlanPer];
  int64_t el = 0, lc = 0;
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    const int b = tid * kPlanPer + k;
    n_el[k] = n_loc[k] = 0;
    if (b < a.batch) {
      const SyncReq q = sync_req(a, b);
      n_el[k] = q.n_patch + q.n_new;
      n_loc[k] = q.n_new;
    }
    el += n_el[k];
    lc += n_loc[k];
  }
  int64_t total, total_loc;
  int64_t e0 = block_scan(el, sm.wsum, total);
  int64_t l0 = block_scan(lc, sm.wsum, total_loc);
#pragma unroll
  for (int k = 0; k < kPlanPer; ++k) {
    sm.flat[tid * kPlanPer + k] = e0;
    sm.loc[tid * kPlanPer + k] = l0;
    e0 += n_el[k];
    l0 += n_loc[k];
  }
  if (tid == 0) sm.flat[kSyncMaxBatch] = total;
  __syncthreads();

  const int64_t step = (int64_t)gridDim.x * kPlanThreads;
  for (int64_t idx = (int64_t)blockIdx.x * kPlanThreads + tid; idx < total; idx += step) {
    int lo = 0, hi = a.batch - 1;   // last request with flat <= idx
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (sm.flat[mid] <= idx) lo = mid; else hi = mid - 1;
    }
    const SyncReq q = sync_req(a, lo);
    const int64_t j = idx - sm.flat[lo];
    int64_t pos, val;
    if (j < q.n_patch) {
      pos = q.pfrom + j;
      val = a.pvals[q.poff + j];
    } else {
      const int64_t li = sm.loc[lo] + (j - q.n_patch);
      if (li >= a.loc_len) continue;
      pos = q.prefix + (j - q.n_patch);
      val = a.loc[li];
    }
    a.table[q.row * a.stride + pos] = val;
  }
}

}  // namespace
}  // namespace tfa

extern "C" {

int64_t tf_attn_plan_device_capacity(int64_t total_tokens, int32_t batch_size,
                                     int32_t num_q_heads, int32_t num_kv_heads) {
  tfa::clear_error();
  if (total_tokens < 0 || batch_size < 0 || num_kv_heads <= 0 || num_q_heads <= 0 ||
      num_q_heads % num_kv_heads)
    return tfa::fail(TF_ERR_INVALID, "plan_device_capacity: bad arguments");
  const int64_t g = num_q_heads / num_kv_heads;
  return (int64_t)num_kv_heads *
         ((total_tokens * g + tfa::kExtendItemRows - 1) / tfa::kExtendItemRows + batch_size);
}

int32_t tf_attn_plan_device(const int64_t* extend_lens, int32_t batch_size,
                            int32_t num_q_heads, int32_t num_kv_heads,
                            int32_t decode_to_decode_kernel, int32_t* work,
                            int32_t work_capacity, int32_t* dec_items, int32_t* dec_rows,
                            int32_t dec_capacity, int32_t* status, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  if (batch_size < 0 || batch_size > kPlanMaxBatch)
    return fail(TF_ERR_UNSUPPORTED, "plan_device: batch_size=%d (at most %d)", batch_size,
                kPlanMaxBatch);
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return fail(TF_ERR_INVALID, "plan_device: heads %d/%d", num_q_heads, num_kv_heads);
  if (work_capacity < 0 || dec_capacity < 0 || !status ||
      (batch_size > 0 && !extend_lens) || (work_capacity > 0 && !work) ||
      (dec_capacity > 0 && (!dec_items || !dec_rows)))
    return fail(TF_ERR_INVALID, "plan_device: null pointer or negative capacity");
  PlanArgs a;
  a.ext = extend_lens;
  a.batch = batch_size;
  a.hkv = num_kv_heads;
  a.group = num_q_heads / num_kv_heads;
  a.dec_to_dec = decode_to_decode_kernel ? 1 : 0;
  a.work = work;
  a.work_cap = work_capacity;
  a.dec_items = dec_items;
  a.dec_rows = dec_rows;
  a.dec_cap = dec_capacity;
  a.status = status;
  hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(kPlanThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  return launch_status("tf_attn_plan_device launch");
}

int32_t tf_attn_plan_blocks(const int32_t* work, int32_t n_work, const int32_t* dec_items,
                            const int32_t* dec_rows, int32_t n_dec, int32_t num_q_heads,
                            int32_t num_kv_heads, int32_t row_groups, int64_t max_rows,
                            int32_t* blocks, int32_t n_blocks, int32_t* pieces,
                            int32_t n_pieces, int32_t* merges, int32_t n_merges,
                            const int64_t* seq_lens, int32_t seq_len_override,
                            int64_t rtt_cols, int32_t key_bytes, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return fail(TF_ERR_INVALID, "plan_blocks: heads %d/%d", num_q_heads, num_kv_heads);
  if (row_groups != 1 && row_groups != 2)
    return fail(TF_ERR_INVALID, "plan_blocks: row_groups=%d (1 or 2)", row_groups);
  if (n_work < 0 || n_dec < 0 || n_blocks < 0 || n_pieces < 0 || (n_work > 0 && !work) ||
      (n_dec > 0 && (!dec_items || !dec_rows)) || (n_blocks > 0 && !blocks) ||
      (n_pieces > 0 && !pieces) || !aligned16(blocks) || !aligned16(pieces) ||
      !aligned16(merges) || n_merges < 0)
    return fail(TF_ERR_INVALID, "plan_blocks: null or misaligned pointer or negative count");
  const int32_t cus = device_cu_count();
  if (merges && (n_pieces < cus || n_merges < 1 || rtt_cols < 1 || key_bytes < 0 ||
                 (!seq_lens && seq_len_override <= 0)))
    return fail(TF_ERR_INVALID, "plan_blocks: a split needs the lengths and room for %d pieces "
                "and 1 merge", cus);
  BlockArgs a;
  a.work = work;
  a.n_work = n_work;
  a.dec_items = dec_items;
  a.dec_rows = dec_rows;
  a.n_dec = n_dec;
  a.group = num_q_heads / num_kv_heads;
  a.unit_rows = 16 * row_groups;
  a.max_rows = max_rows;
  a.blocks = reinterpret_cast<RowItem*>(blocks);
  a.n_blocks = n_blocks;
  a.pieces = pieces;
  a.n_pieces = n_pieces;
  a.merges = merges;
  a.n_merges = n_merges;
  a.seq_lens = seq_lens;
  a.seq_override = seq_len_override;
  a.rtt_cols = rtt_cols;
  a.key_bytes = key_bytes;
  a.cus = cus;
  hipLaunchKernelGGL(blocks_kernel, dim3(1), dim3(kPlanThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  return launch_status("tf_attn_plan_blocks launch");
}

int32_t tf_req_to_token_sync(int64_t* req_to_token, int64_t rtt_rows, int64_t rtt_row_stride,
                             int64_t rtt_cols, const int64_t* req_pool_indices,
                             const int64_t* prefix_lens, const int64_t* seq_lens,
                             const int64_t* out_cache_loc, int64_t out_cache_loc_len,
                             const int64_t* patch_from, const int64_t* patch_offsets,
                             const int64_t* patch_vals, int64_t patch_vals_len,
                             int32_t batch_size, int32_t num_workgroups, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  if (batch_size < 0 || batch_size > kSyncMaxBatch)
    return fail(TF_ERR_UNSUPPORTED, "req_to_token_sync: batch_size=%d (at most %d)",
                batch_size, kSyncMaxBatch);
  if (num_workgroups < 0 || num_workgroups > 4096)
    return fail(TF_ERR_INVALID, "req_to_token_sync: num_workgroups=%d", num_workgroups);
  if (batch_size == 0) return TF_OK;
  if (!req_to_token || !req_pool_indices || !prefix_lens || !seq_lens)
    return fail(TF_ERR_INVALID, "req_to_token_sync: null pointer argument");
  if (rtt_rows < 1 || rtt_cols < 1 || rtt_row_stride < rtt_cols)
    return fail(TF_ERR_INVALID, "req_to_token_sync: table %lld x %lld, row stride %lld",
                (long long)rtt_rows, (long long)rtt_cols, (long long)rtt_row_stride);
  if (out_cache_loc_len < 0 || (out_cache_loc_len > 0 && !out_cache_loc))
    return fail(TF_ERR_INVALID, "req_to_token_sync: out_cache_loc of %lld entries",
                (long long)out_cache_loc_len);
  const bool patches = patch_from || patch_offsets || patch_vals;
  if (patches && (!patch_from || !patch_offsets || (patch_vals_len > 0 && !patch_vals)))
    return fail(TF_ERR_INVALID,
                "req_to_token_sync: patch_from, patch_offsets and patch_vals go together");
  if (patch_vals_len < 0)
    return fail(TF_ERR_INVALID, "req_to_token_sync: patch_vals_len=%lld",
                (long long)patch_vals_len);
  SyncArgs a;
  a.table = req_to_token;
  a.rows = rtt_rows;
  a.stride = rtt_row_stride;
  a.cols = rtt_cols;
  a.rpi = req_pool_indices;
  a.prefix = prefix_lens;
  a.seq = seq_lens;
  a.loc = out_cache_loc;
  a.loc_len = out_cache_loc_len;
  a.pfrom = patches ? patch_from : nullptr;
  a.poff = patches ? patch_offsets : nullptr;
  a.pvals = patches ? patch_vals : nullptr;
  a.pvals_len = patches ? patch_vals_len : 0;
  a.batch = batch_size;
  hipLaunchKernelGGL(rtt_sync_kernel, dim3(num_workgroups ? num_workgroups : 64),
                     dim3(kPlanThreads), 0, reinterpret_cast<hipStream_t>(stream), a);
  return launch_status("tf_req_to_token_sync launch");
}

}  // extern "C"
