// Decode attention over the req_to_token -> KV-pool slot indirection.
//
// Replaces the reference's pure-decode branch (qwen3_8/full_attention.py:215-242):
// gather of req_to_token[r, :L] rows, GQA repeat_interleave, length mask and
// SDPA, here fused into one HBM-streaming pass with no padded or expanded copy.
//
// Work decomposition (persistent, balanced)
//   unit = (request item, kv head, group of <= 16 q heads sharing that kv head);
//   a unit's context is cut into 16-token tiles, and the tiles of all units,
//   laid out unit after unit, form one global range of N tiles. The grid has
//   P = one workgroup per CU (all resident at once); workgroup b owns global
//   tiles [floor(b N / P), floor((b+1) N / P)), so every CU gets the same work
//   whatever the length mix. A workgroup walks its range as segments (one unit
//   each); 4 waves take interleaved tiles of a segment. A unit owned entirely by
//   one workgroup is written as final bf16 output; otherwise each owner stores
//   an fp32 partial (O, max, sum) and a second small kernel merges them.  Only a
//   workgroup's first and last unit can be shared: its partials are at slots 2 b
//   and 2 b + 1, or at b + u (unique, < P + units) where that takes fewer (and in
//   tf_attn_decode, whose workspace has that size).
//   The whole GQA head group of a kv head shares every K/V row read from HBM.
// Per segment: the slot ids of up to 2048 tokens at a time (int64 req_to_token
// entries clamped to the pool) are staged in LDS with coalesced loads, and the
// group's Q^T MFMA fragments once.
// Per 16-token tile a wave
//   * loads K and V rows with the same row-contiguous pattern (lane (g, n) reads
//     16-byte chunk n (+16) of the rows of tokens 4g + j) using nontemporal
//     loads; the next tile's K is issued as soon as this tile's K is staged and
//     its V as soon as PV has consumed this tile's V, so a tile's worth of loads
//     is always in flight per wave,
//   * stages K through a per-wave, XOR-swizzled LDS tile into the MFMA
//     A-operand layout (row = lane % 16), conflict-free both ways,
//   * S^T[token, head] = K * Q^T with v_mfma_f32_16x16x32_bf16 (heads padded to 16),
//   * online softmax per head (lane-local scores, two xor-shuffles for the max),
//   * O^T[dim, head] += V^T * P^T with v_mfma_f32_16x16x16_bf16, V^T built in
//     registers with v_perm_b32 (fp8: byte permutes + v_cvt_scalef32_pk_bf16_fp8).
//   Every per-head quantity (max, sum, rescale factor, 64 output dims) is then
//   lane-local: lane (g, n) owns head n, dims {128s + 32g + 8r + e} (bf16) or
//   {64g + 16r + e} (fp8).
// Row blocks (tf_attn_rows).  The same kernel takes several query rows per
// unit: the (token, head) rows of a request with few new tokens, or blocks of 32
// rows of any request at head dims other than 256.  Up to two groups of 16 rows
// share every K / V tile a wave loads, each row masked at its own last key; the
// group's softmax state and 64 (or 32) output dims per lane are all that grows.
// 20 requests of 2 to 4 tokens on 1k to 8k keys stream 362 MB in 76 us.
// The merge lives in its own launch so the streaming kernel needs no
// device-scope fence (on gfx950 those write back and invalidate the XCD's L2).
#include <math.h>

#include <mutex>

#include "attn_row.h"
#include "tf_common.h"
#include "tf_internal.h"

namespace tfa {
namespace {

constexpr int kD = 256;         // head_dim (Qwen3.8: 256)
constexpr int kWaves = 4;
constexpr int kTile = 16;       // tokens per wave iteration
constexpr int kMaxChunk = 2048; // slot ids staged in LDS at a time
constexpr int kMaxItems = 2048; // requests per launch (per-item prefix lives in LDS)

struct DecodeArgs {
  const __bf16* q;
  int64_t q_stride;
  const uint8_t* k_pool;
  const uint8_t* v_pool;
  int64_t pool_slots;
  const float* k_scale;
  const float* v_scale;
  const int64_t* rtt;
  int64_t rtt_rows, rtt_stride, rtt_cols;
  const int64_t* rpi;
  const int64_t* seq_lens;
  int32_t seq_override;
  const int32_t* items;    // batch index of each item (-1: padding) and its q row;
  const int32_t* q_rows;   //   NULL: item i is request i, row i
  const RowItem* blocks;   // or: row blocks (several query rows of a request each)
  int32_t n_items;
  int32_t hkv, group, n_hg;
  int32_t head_dim;
  float scale_log2;
  __bf16* out;
  int64_t out_stride;
  const __bf16* gate;   // optional output gate (NULL: none)
  int64_t gate_stride, gate_hstride;
  uint32_t* amax;       // optional: raised to max |out| (bf16 bits), amax_commit
  float* ws_ml;
  float* ws_o;
  int32_t* ipre;      // row plans: the streaming kernel's tile prefix, for the merge
  int32_t* odd;       // OTHER: per unit that one workgroup owns, whether its O is not finite
  int32_t n_blocks;   // P: workgroups of the streaming kernel
  bool by_owner;      // partial slots: two per workgroup (else one per workgroup and unit)
};

// The kernels' shape.  DP: head dims in a row's tile (256, or 128 for head dims up
// to 128); NG: groups of 16 query rows a unit holds (1 or 2: four groups of 256 dims
// spill); OTHER: head dims that do not fill the tile (chunks past the head dim are
// read as zeros and not written) and probabilities split into three bf16 parts, all
// of their 24 bits, which the PV product takes one after the other, smallest first
// (the kernel these head dims ran before kept them in fp32; two parts are off by up
// to 2^-18 and 1 to 5 % faster).  BLK: items are row blocks (DecodeArgs::blocks);
// else one token each, and every row sees every key of its item.
template <int DP_, bool FP8_, int NG_, bool OTHER_, bool BLK_>
struct Cfg {
  static constexpr int DP = DP_;
  static constexpr bool FP8 = FP8_;
  static constexpr int NG = NG_;
  static constexpr bool OTHER = OTHER_;
  static constexpr bool BLK = BLK_;
  static_assert(DP == 256 || (DP == 128 && !FP8), "tile width");
  static constexpr int kAcc = DP / 16;                 // f32x4 accumulators per lane and group
  static constexpr int kChunks = FP8 ? 16 : DP / 8;    // 16-byte chunks per row of the tile
  static constexpr int kS = kChunks / 16;              // chunks per lane and token
  static constexpr int kSteps = DP / 32;               // 32-dim MFMA steps of QK^T
  static constexpr int kRows = 16 * NG;                // query rows per unit
  static constexpr int kRowFloats = DP;                // a partial row's O
  static constexpr bool kRowPlan = OTHER || BLK;       // DecodeArgs::by_owner and ipre are set
};

template <class C>
struct WaveState {
  float m[C::NG], l[C::NG];
  f32x4 acc[C::NG][C::kAcc];
};

// LDS slot for one group of one wave's state, element-major so lanes hit
// consecutive banks.
template <class C>
struct StateSlot {
  f32x4 acc[C::kAcc][kWave];
  float m[kWave];
  float l[kWave];
};

// Per-wave K staging tile: 16 token rows x kChunks 16-byte chunks; chunk c of
// row r sits at r * kChunks + (c ^ r) so that both the coalesced writes and the
// MFMA-layout reads are free of bank conflicts.
template <class C>
struct DecodeSmem {
  union {
    struct {
      int32_t slots[kMaxChunk];                     // slot id of each staged token
      u32x4 kstage[kWaves][kTile * C::kChunks];     // per-wave K tile
    } loop;
    StateSlot<C> merge[2];                          // wave-state exchange
  } u;
  u32x4 qfrag[C::NG][C::kSteps][kWave];             // Q^T B-operand fragments, lane-major
  int32_t ipre[kMaxItems + 1];                      // exclusive prefix of per-item tiles
  int32_t wsum[kWaves];
};

// Per-lane register slices of one 16-token tile: K (staged to LDS for the
// S^T = K Q^T MFMA) and V (transposed in registers for the PV MFMA).
template <class C>
struct KBuf {
  u32x4 k[4][C::kS];   // row of token 4g + j, chunk n + 16 s
};
template <class C>
struct VBuf {
  u32x4 v[4][C::kS];
};

template <class C>
__device__ __forceinline__ void merge_into(WaveState<C>& st, int q, float m2, float l2,
                                           const f32x4* acc2) {
  const float M = fmaxf(st.m[q], m2);
  const float a1 = (st.m[q] == -INFINITY) ? 0.f : fast_exp2(st.m[q] - M);
  const float a2 = (m2 == -INFINITY) ? 0.f : fast_exp2(m2 - M);
  st.l[q] = st.l[q] * a1 + l2 * a2;
#pragma unroll
  for (int i = 0; i < C::kAcc; ++i) st.acc[q][i] = st.acc[q][i] * a1 + acc2[i] * a2;
  st.m[q] = M;
}

template <class C>
__device__ __forceinline__ void reset_state(WaveState<C>& st) {
#pragma unroll
  for (int q = 0; q < C::NG; ++q) {
    st.m[q] = -INFINITY;
    st.l[q] = 0.f;
#pragma unroll
    for (int i = 0; i < C::kAcc; ++i) st.acc[q][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

template <class C>
__device__ __forceinline__ void put_state(StateSlot<C>* s, int lane, const WaveState<C>& st,
                                          int q) {
#pragma unroll
  for (int i = 0; i < C::kAcc; ++i) s->acc[i][lane] = st.acc[q][i];
  s->m[lane] = st.m[q];
  s->l[lane] = st.l[q];
}

template <class C>
__device__ __forceinline__ void take_state(const StateSlot<C>* s, int lane, WaveState<C>& st,
                                           int q) {
  f32x4 acc2[C::kAcc];
#pragma unroll
  for (int i = 0; i < C::kAcc; ++i) acc2[i] = s->acc[i][lane];
  merge_into<C>(st, q, s->m[lane], s->l[lane], acc2);
}

// Tree merge of the 4 wave states, group by group; wave 0 ends up holding the
// block state.
template <class C>
__device__ __forceinline__ void block_merge(StateSlot<C>* slots, int w, int lane,
                                            WaveState<C>& st, int n_groups) {
#pragma unroll
  for (int q = 0; q < C::NG; ++q) {
    if (C::NG > 1 && q >= n_groups) break;
    __syncthreads();
    if (w >= 2) put_state<C>(&slots[w - 2], lane, st, q);
    __syncthreads();
    if (w < 2) take_state<C>(&slots[w], lane, st, q);
    __syncthreads();
    if (w == 1) put_state<C>(&slots[0], lane, st, q);
    __syncthreads();
    if (w == 0) take_state<C>(&slots[0], lane, st, q);
  }
}

// Writes group q of the state; returns the largest |value| written (bf16 bits)
// for amax_commit.  A row that saw no key (l = 0) is zeros.
template <class C>
__device__ __forceinline__ uint32_t write_output(const DecodeArgs& a, int qrow, int hq, int g,
                                                 const WaveState<C>& st, int q, float vscale) {
  const float inv = st.l[q] > 0.f || st.l[q] != st.l[q] ? vscale / st.l[q] : 0.f;
  uint32_t m = 0;
  const int D = C::OTHER ? a.head_dim : C::DP;
  __bf16* o = a.out + (int64_t)qrow * a.out_stride + (int64_t)hq * D;
  const __bf16* gt =
      a.gate ? a.gate + (int64_t)qrow * a.gate_stride + (int64_t)hq * a.gate_hstride : nullptr;
  // 8 outputs (dims off .. off + 7) per store; gated when the caller passed one.
  auto store8 = [&](int off, u32x4 v) {
    if (C::OTHER && off >= D) return;
    if (gt) {
      const u32x4 gv = ld_g16(gt + off);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = gate_pair(v[k], gv[k]);
    }
    m = max(m, abs_max8(v));
    *reinterpret_cast<u32x4*>(o + off) = v;
  };
  const f32x4* acc = st.acc[q];
  if (C::FP8) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = pack_bf16(acc[8 * h + 2 * k][r] * inv, acc[8 * h + 2 * k + 1][r] * inv);
        store8(64 * g + 16 * r + 8 * h, v);
      }
    }
  } else {
#pragma unroll
    for (int s = 0; s < C::kS; ++s) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        u32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          v[k] = pack_bf16(acc[8 * s + 2 * k][r] * inv, acc[8 * s + 2 * k + 1][r] * inv);
        store8(128 * s + 32 * g + 8 * r, v);
      }
    }
  }
  return m;
}

// Issue the loads of tile `it` (chunk tokens it*16 .. it*16+15, clamped to the
// chunk's last token so every address is a valid row): lane (g, n) reads chunk
// n (+ 16 s) of the rows of tokens 4g + j, the same row-contiguous pattern for
// K (the MFMA layout is produced through LDS) and V.  The loads are nontemporal:
// one-token units stream every row once.  Blocks of one request read its rows
// again, each for itself, and plain loads serve those better (2 prompts beside 12
// decodes at 128 dims 94.8 and 84.2 us, 20 requests of 6 tokens at 256 153 and 143),
// but cost steps of many rows that are read once more (64 decodes beside 3 tokens
// 211 and 240, 64 requests of 5 tokens 232 and 256).  n_chunks: chunks of a row
// (OTHER).
template <class C>
__device__ __forceinline__ void issue_rows(u32x4 (&x)[4][C::kS], const int32_t* slots, int it,
                                           int n_loc, int g, int n, const uint8_t* base,
                                           int64_t slot_bytes, int n_chunks) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t sl = slots[min(it * kTile + 4 * g + j, n_loc - 1)];
    const uint8_t* p = base + sl * slot_bytes;
#pragma unroll
    for (int s = 0; s < C::kS; ++s) {
      if (C::OTHER)
        x[j][s] = n + 16 * s < n_chunks ? ld_nt16(p + 16 * n + 256 * s) : u32x4{0u, 0u, 0u, 0u};
      else
        x[j][s] = ld_nt16(p + 16 * n + 256 * s);
    }
  }
}

// Writes the tile's K chunks to this wave's LDS staging tile (swizzled).
template <class C>
__device__ __forceinline__ void stage_k(const KBuf<C>& kb, u32x4* ks, int g, int n) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = 4 * g + j;
#pragma unroll
    for (int s = 0; s < C::kS; ++s) ks[r * C::kChunks + ((n + 16 * s) ^ r)] = kb.k[j][s];
  }
}

// The staged tile's K fragments, bf16: k-step kk of lane (g, n) is row n, dims
// 32kk + 8g .. (bf16: chunk 4kk + g) or, for fp8, dims 64u + 16g .. (chunk
// 4u + g, two k-steps).
template <class C>
__device__ __forceinline__ void k_frags(const u32x4* ks, int g, int n, u32x4 (&kf)[C::kSteps]) {
  if (C::FP8) {
#pragma unroll
    for (int u = 0; u < C::kSteps / 2; ++u) {
      const u32x4 x = ks[n * 16 + ((4 * u + g) ^ n)];
      kf[2 * u] = e4m3x8_to_bf16x8(x[0], x[1]);
      kf[2 * u + 1] = e4m3x8_to_bf16x8(x[2], x[3]);
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < C::kSteps; ++kk) kf[kk] = ks[n * C::kChunks + ((4 * kk + g) ^ n)];
  }
}

// S^T = K Q^T for the tile, then the online-softmax update of group q's row n,
// whose visible tokens are those below lim (chunk-local); returns the tile's
// probabilities packed as the PV B operand (P^T, 4 tokens per lane), pl their
// lower parts, smallest first (OTHER).
template <class C>
__device__ __forceinline__ u32x2 qk_softmax(const u32x4 (&kf)[C::kSteps],
                                            const u32x4 (&qf)[C::kSteps], int it, int lim, int g,
                                            float sl2, WaveState<C>& st, int q,
                                            u32x2 (&pl)[2]) {
  f32x4 sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < C::kSteps; ++kk) sacc = mfma_16x16x32(kf[kk], qf[kk], sacc);
  float sc[4];
  float mx = -INFINITY;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = it * kTile + 4 * g + r;
    sc[r] = (t < lim) ? sacc[r] * sl2 : -INFINITY;
    mx = fmaxf(mx, sc[r]);
  }
  mx = wave_max_xor(mx, 16);
  mx = wave_max_xor(mx, 32);
  const float mnew = fmaxf(st.m[q], mx);
  // A causal row may not have seen a key yet: exponents relative to 0 then.
  const float mref = C::BLK && mnew == -INFINITY ? 0.f : mnew;
  const float alpha = fast_exp2(st.m[q] - mref);
  float p[4];
  float psum = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    p[r] = fast_exp2(sc[r] - mref);
    psum += p[r];
  }
  st.l[q] = st.l[q] * alpha + psum;
  st.m[q] = mnew;
  if (__ballot(alpha != 1.f)) {
#pragma unroll
    for (int i = 0; i < C::kAcc; ++i) st.acc[q][i] *= alpha;
  }
  const u32x2 ph = {pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
  if (C::OTHER) {   // (the differences are exact)
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] -= r & 1 ? bf16_hi(ph[r >> 1]) : bf16_lo(ph[r >> 1]);
    pl[1] = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] -= r & 1 ? bf16_hi(pl[1][r >> 1]) : bf16_lo(pl[1][r >> 1]);
    pl[0] = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
  }
  return ph;
}

// O^T += V^T P^T for the tile, every group.
template <class C>
__device__ __forceinline__ void pv(const VBuf<C>& vb, const u32x2 (&pt)[C::NG],
                                   const u32x2 (&pl)[C::NG][2], WaveState<C>& st,
                                   int n_groups) {
  auto mma = [&](int i, u32x2 va) {
#pragma unroll
    for (int q = 0; q < C::NG; ++q) {
      if (C::NG > 1 && q >= n_groups) break;
      if (C::OTHER) {
#pragma unroll
        for (int k = 0; k < 2; ++k) st.acc[q][i] = mfma_16x16x16(va, pl[q][k], st.acc[q][i]);
      }
      st.acc[q][i] = mfma_16x16x16(va, pt[q], st.acc[q][i]);
    }
  };
  if (C::FP8) {
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const int dw = e >> 2;
      const uint32_t b0 = e & 3;
      const uint32_t sel = b0 | ((4 + b0) << 8) | ((b0 + 1) << 16) | ((5 + b0) << 24);
      const uint32_t x = __builtin_amdgcn_perm(vb.v[1][0][dw], vb.v[0][0][dw], sel);
      const uint32_t y = __builtin_amdgcn_perm(vb.v[3][0][dw], vb.v[2][0][dw], sel);
      mma(e, u32x2{e4m3x2_to_bf16x2<false>(x), e4m3x2_to_bf16x2<false>(y)});
      mma(e + 1, u32x2{e4m3x2_to_bf16x2<true>(x), e4m3x2_to_bf16x2<true>(y)});
    }
  } else {
#pragma unroll
    for (int s = 0; s < C::kS; ++s) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int dw = e >> 1;
        const int hi = e & 1;
        mma(8 * s + e, u32x2{pair_sel(vb.v[1][s][dw], vb.v[0][s][dw], hi),
                             pair_sel(vb.v[3][s][dw], vb.v[2][s][dw], hi)});
      }
    }
  }
}

__device__ __forceinline__ bool not_finite(const f32x4& v) {
  float y = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) y = fmaf(v[e], 0.f, y);
  return y != y;
}

// Whether any of the lane's accumulators is NaN or infinite.
template <class C>
__device__ __forceinline__ bool any_odd(const WaveState<C>& st) {
  f32x4 x[2] = {};   // (eight short chains)
#pragma unroll
  for (int q = 0; q < C::NG; ++q)
#pragma unroll
    for (int i = 0; i < C::kAcc; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[i & 1][e] = fmaf(st.acc[q][i][e], 0.f, x[i & 1][e]);
  const float y = (x[0][0] + x[0][1] + x[0][2] + x[0][3]) + (x[1][0] + x[1][1] + x[1][2] + x[1][3]);
  return y != y;
}

// Item i of the call: query rows row0 .. (row = t * G + h: token t of the
// request's ext new tokens, head h of the kv head's group) of request b, whose
// first token is q row qrow.  A negative b marks a padding entry of a
// device-built list: no work and no output.
template <class C>
__device__ __forceinline__ RowItem item_of(const DecodeArgs& a, int i) {
  if (C::BLK) return a.blocks[i];
  const int b = a.items ? a.items[i] : i;
  return RowItem{b, a.q_rows ? a.q_rows[i] : b, 1, 0};
}

// Context length of the item's request (its seq_len, or the bsz == 1
// override), clamped to the req_to_token row.
__device__ __forceinline__ int item_len(const DecodeArgs& a, const RowItem& it) {
  if (it.b < 0) return 0;
  int64_t len = a.seq_override > 0 ? (int64_t)a.seq_override : a.seq_lens[it.b];
  if (len > a.rtt_cols) len = a.rtt_cols;
  return len > 0 ? (int)len : 0;
}

// Keys the item reads: up to the last one that its last row sees.
template <class C>
__device__ __forceinline__ int item_keys(const DecodeArgs& a, const RowItem& it) {
  const int len = item_len(a, it);
  if (!C::BLK) return len;
  const int last = min(it.row0 + C::kRows, it.ext * a.group) - 1;
  return max(0, min(len, len - it.ext + last / a.group + 1));
}

template <class C>
__device__ __forceinline__ int item_tiles(const DecodeArgs& a, int i) {
  return (item_keys<C>(a, item_of<C>(a, i)) + kTile - 1) / kTile;
}

// ipre[i] = sum of tiles of items < i, ipre[n_items] = total (block-wide scan).
template <class C>
__device__ void item_prefix(const DecodeArgs& a, int32_t* ipre, int32_t* wsum) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = wave_id();
  constexpr int kPer = kMaxItems / (kWaves * kWave);
  int t[kPer];
  int sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    t[k] = i < a.n_items ? item_tiles<C>(a, i) : 0;
    sum += t[k];
  }
  int incl = sum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int v = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += v;
  }
  if (lane == kWave - 1) wsum[w] = incl;
  __syncthreads();
  int excl = incl - sum;
  for (int k = 0; k < w; ++k) excl += wsum[k];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = tid * kPer + k;
    if (i <= a.n_items) ipre[i] = excl;
    excl += t[k];
  }
  if (tid == kWaves * kWave - 1 && a.n_items == kMaxItems) ipre[kMaxItems] = excl;
  __syncthreads();
}

// Workgroup that owns global tile x when N tiles are split over P workgroups.
__device__ __forceinline__ int owner_of(int64_t x, int64_t N, int P) {
  return (int)(((x + 1) * P - 1) / N);
}

// Units of 16 query rows, and of 128 dims, run two workgroups per CU where the
// grid has more than one per CU; the accumulators of 32 rows of 256 dims fill
// the registers of one.
template <class C>
__global__ void __launch_bounds__(kWaves * kWave, C::NG == 1 || C::DP == 128 ? 2 : 1)
decode_kernel(DecodeArgs a) {
  __shared__ DecodeSmem<C> sm;
  const int D = C::OTHER ? a.head_dim : C::DP;
  const int row_bytes = C::FP8 ? D : 2 * D;
  const int n_chunks = row_bytes / 16;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = wave_id();
  const int g = lane >> 4;
  const int n = lane & 15;

  item_prefix<C>(a, sm.ipre, sm.wsum);
  if (C::kRowPlan && blockIdx.x == 0)
    for (int i = tid; i <= a.n_items; i += kWaves * kWave) a.ipre[i] = sm.ipre[i];
  const int units_per_item = a.hkv * a.n_hg;
  const int64_t N = (int64_t)units_per_item * sm.ipre[a.n_items];
  // With P <= N every workgroup's range is non-empty, so the owners of a unit
  // are consecutive workgroups (the merge kernel relies on it).
  const int P = (int)min<int64_t>(a.n_blocks, N);
  if ((int)blockIdx.x >= P) return;
  const int64_t x_end = (int64_t)(blockIdx.x + 1) * N / P;
  int64_t x = (int64_t)blockIdx.x * N / P;

  const float kscale = C::FP8 ? a.k_scale[0] : 1.f;
  const float vscale = C::FP8 ? a.v_scale[0] : 1.f;
  const float sl2 = a.scale_log2 * kscale;
  const int64_t slot_bytes = (int64_t)a.hkv * row_bytes;

  // First item whose tile range contains x (binary search over ipre).
  int item = 0;
  {
    int lo = 0, hi = a.n_items - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if ((int64_t)units_per_item * sm.ipre[mid] <= x) lo = mid; else hi = mid - 1;
    }
    item = lo;
  }

  for (int part_at = 0; x < x_end; part_at = 1) {   // 0: the workgroup's first unit
    // ---- locate the segment: unit (item, j), tiles [t0, t1)
    while ((int64_t)units_per_item * sm.ipre[item + 1] <= x) ++item;
    const int Ti = sm.ipre[item + 1] - sm.ipre[item];
    const int64_t r = x - (int64_t)units_per_item * sm.ipre[item];
    const int j = (int)(r / Ti);
    const int t0 = (int)(r - (int64_t)j * Ti);
    const int t1 = (int)min<int64_t>(Ti, t0 + (x_end - x));
    x += t1 - t0;

    const int hk = j / a.n_hg;
    const int hg = j - hk * a.n_hg;
    const RowItem im = item_of<C>(a, item);
    const int len = item_len(a, im), L = item_keys<C>(a, im);
    const int unit_row = im.row0 + hg * C::kRows;          // the unit's first row
    const int n_rows = im.ext * a.group - unit_row;        // its rows (of kRows)
    const int n_groups = min((n_rows + 15) / 16, C::NG);
    const int64_t row = clamp_i64(a.rpi[im.b], 0, a.rtt_rows - 1);
    const int64_t* rtt = a.rtt + row * a.rtt_stride;
    const uint8_t* kbase = a.k_pool + (int64_t)hk * row_bytes;
    const uint8_t* vbase = a.v_pool + (int64_t)hk * row_bytes;
    // Row n of group q: its q row and head, and how many keys it sees.
    auto row_of = [&](int q, int& qrow, int& hq, int& seen) {
      const int rho = min(unit_row + 16 * q + n, im.ext * a.group - 1);
      const int t = C::BLK ? rho / a.group : 0;
      qrow = im.qrow + t;
      hq = hk * a.group + rho - t * a.group;
      seen = C::BLK ? len - im.ext + t + 1 : len;
      return 16 * q + n < n_rows;
    };
    int seen[C::NG];
#pragma unroll
    for (int q = 0; q < C::NG; ++q) {
      int qrow, hq;
      row_of(q, qrow, hq, seen[q]);
    }

    WaveState<C> st;
    reset_state<C>(st);
    for (int sub = t0; sub < t1; sub += kMaxChunk / kTile) {
      const int c0 = sub * kTile;
      const int n_loc = min(L, min(t1, sub + kMaxChunk / kTile) * kTile) - c0;
      const int n_tiles = (n_loc + kTile - 1) / kTile;
      // ---- stage the slot ids (and, once per segment, the Q^T fragments)
      __syncthreads();
      for (int i = tid; i < n_loc; i += kWaves * kWave)
        sm.u.loop.slots[i] = (int32_t)pool_row(rtt[c0 + i], a.pool_slots, a.seq_override > 0);
      if (sub == t0) {
#pragma unroll
        for (int q = 0; q < C::NG; ++q) {
          if (w != q % kWaves || q >= n_groups) continue;
          int qrow, hq, s;
          const bool ok = row_of(q, qrow, hq, s);
          const __bf16* qp = a.q + (int64_t)qrow * a.q_stride + (int64_t)hq * D;
#pragma unroll
          for (int kk = 0; kk < C::kSteps; ++kk) {
            const int d0 = C::FP8 ? (64 * (kk >> 1) + 16 * g + 8 * (kk & 1)) : (32 * kk + 8 * g);
            sm.qfrag[q][kk][lane] =
                ok && (!C::OTHER || d0 < D) ? ld_g16(qp + d0) : u32x4{0u, 0u, 0u, 0u};
          }
        }
      }
      __syncthreads();

      // ---- this wave's tiles (it = w, w+4, ...): K of the next tile is issued
      // once this tile's K is staged, V of the next tile once PV has consumed
      // this tile's V. The steady-state loop always has a next tile; the last
      // tile is peeled so every wait count is exact.
      int it = w;
      if (it < n_tiles) {
        u32x4 qf[C::kSteps];
        if (C::NG == 1) {
#pragma unroll
          for (int kk = 0; kk < C::kSteps; ++kk) qf[kk] = sm.qfrag[0][kk][lane];
        }
        KBuf<C> kb;
        VBuf<C> vb;
        const int32_t* slots = sm.u.loop.slots;
        u32x4* ks = sm.u.loop.kstage[w];
        auto scores = [&](int it, u32x2 (&pt)[C::NG], u32x2 (&pl)[C::NG][2]) {
          u32x4 kf[C::kSteps];
          k_frags<C>(ks, g, n, kf);
#pragma unroll
          for (int q = 0; q < C::NG; ++q) {
            if (C::NG > 1) {
              if (q >= n_groups) break;
        #pragma unroll
              for (int kk = 0; kk < C::kSteps; ++kk) qf[kk] = sm.qfrag[q][kk][lane];
            }
            const int lim = C::BLK ? min(n_loc, seen[q] - c0) : n_loc;
            pt[q] = qk_softmax<C>(kf, qf, it, lim, g, sl2, st, q, pl[q]);
          }
        };
        u32x2 pt[C::NG], pl[C::NG][2];
        issue_rows<C>(kb.k, slots, it, n_loc, g, n, kbase, slot_bytes, n_chunks);
        issue_rows<C>(vb.v, slots, it, n_loc, g, n, vbase, slot_bytes, n_chunks);
        for (; it + kWaves < n_tiles; it += kWaves) {
          stage_k<C>(kb, ks, g, n);
          // Scheduling barriers keep each prefetch where it is: the scheduler
          // would otherwise sink it to just before its consumer.
          __builtin_amdgcn_sched_barrier(0);
          issue_rows<C>(kb.k, slots, it + kWaves, n_loc, g, n, kbase, slot_bytes, n_chunks);
          __builtin_amdgcn_sched_barrier(0);
          scores(it, pt, pl);
          pv<C>(vb, pt, pl, st, n_groups);
          __builtin_amdgcn_sched_barrier(0);
          issue_rows<C>(vb.v, slots, it + kWaves, n_loc, g, n, vbase, slot_bytes, n_chunks);
          __builtin_amdgcn_sched_barrier(0);
        }
        stage_k<C>(kb, ks, g, n);
        scores(it, pt, pl);
        pv<C>(vb, pt, pl, st, n_groups);
      }
    }

    // Row sums were accumulated per lane group; the 4 groups share one head.
#pragma unroll
    for (int q = 0; q < C::NG; ++q) {
      st.l[q] += __shfl_xor(st.l[q], 16, kWave);
      st.l[q] += __shfl_xor(st.l[q], 32, kWave);
    }
    block_merge<C>(sm.u.merge, w, lane, st, n_groups);

    if (w == 0) {
      const bool whole = t0 == 0 && t1 == Ti;
      if constexpr (C::OTHER) {
        // NaN or infinite V values: the merge does such a unit's rows again, and
        // writes them and their amax (see decode_merge_kernel).
        if (whole) {
          const bool odd = __ballot(any_odd<C>(st)) != 0;
          if (lane == 0) a.odd[(int64_t)item * units_per_item + j] = odd;
          if (odd) continue;
        }
      }
      uint32_t om = 0;
#pragma unroll
      for (int q = 0; q < C::NG; ++q) {
        if (q >= n_groups) break;
        int qrow, hq, s;
        const bool ok = row_of(q, qrow, hq, s);
        if (!ok) continue;
        if (whole) {
          om = max(om, write_output<C>(a, qrow, hq, g, st, q, vscale));
        } else {
          // Partial of unit u = item * units_per_item + j from this workgroup.
          const int64_t part = C::kRowPlan && a.by_owner
                                   ? 2 * (int64_t)blockIdx.x + part_at
                                   : (int64_t)blockIdx.x + (int64_t)item * units_per_item + j;
          const int64_t pr = part * C::kRows + 16 * q + n;
          f32x4* po = reinterpret_cast<f32x4*>(a.ws_o + pr * C::kRowFloats) + g * C::kAcc;
#pragma unroll
          for (int i = 0; i < C::kAcc; ++i) po[i] = st.acc[q][i];
          if (g == 0) {
            a.ws_ml[pr * 2 + 0] = st.m[q];
            a.ws_ml[pr * 2 + 1] = st.l[q];
          }
        }
      }
      if (whole) amax_commit(a.amax, om);
    }
  }
}

// Merges the partials of every unit owned by more than one workgroup of the
// streaming kernel.  WPR waves share one (unit, head) row, 256 dims = 4 per
// lane: they take the row's partials in turn, kMergeAhead of them in flight per
// wave, and combine through LDS.  Bound by the latency of those reads.  Few
// units (a small batch) are cut into many partials each (B = 1, 4 kv heads: 64
// per unit), so a row gets a whole workgroup; with many units a row has two or
// three partials and one wave.  One workgroup per unit, each wave walking its
// share of the partials with all heads in registers, took 19.5 us at B = 1
// (1531 keys), 11.7 us at B = 16 (with gate and amax) and 6.2 us at B = 64;
// this takes 6.1, 7.3 and 4.9 us.  Eight waves per workgroup: with four, the
// amax atomics (one per workgroup on one word) took 1.7 us more at B = 16, with
// sixteen a launch starts 2 us later.
// NaN or infinite V values at other head dims (OTHER): an MFMA multiplies every V
// row of a tile with every query row's p, zero for keys the row does not see
// (later tokens, repeats past the last key), and the low part of a visible key's
// p may be zero or negative.  A row whose O is not finite is done again here,
// over the keys it sees: O is looked at once per row or whole unit (a test of
// each tile's V in the streaming kernel took 2 to 40 % of it; the rows done again
// there cost it 3 %, in scalar registers).
// Units of an empty request (L = 0) get zeros, as the reference's fully masked
// scaled_dot_product_attention returns them (torch's safe softmax: a row with
// no visible key is all zeros).
constexpr int kMergeAhead = 8;
constexpr int kMergeWaves = 8;

template <class C, int WPR>
__global__ void __launch_bounds__(kMergeWaves * kWave)
decode_merge_kernel(DecodeArgs a) {
  constexpr int kRows = kMergeWaves / WPR;   // rows of the unit side by side
  __shared__ f32x4 so[kMergeWaves][kWave];   // a wave's O in the partials' order, then dim order
  __shared__ float sm_m[kMergeWaves], sm_l[kMergeWaves];
  __shared__ int32_t red[2][kMergeWaves];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = wave_id();

  const int units_per_item = a.hkv * a.n_hg;
  const int u = blockIdx.x;
  const int item = u / units_per_item;
  const int j = u - item * units_per_item;
  const int hk = j / a.n_hg;
  const RowItem im = item_of<C>(a, item);
  const int unit_row = im.row0 + (j - hk * a.n_hg) * C::kRows;
  const int n_rows = min(im.ext * a.group - unit_row, C::kRows);   // the unit's rows
  const int first = blockIdx.y * kRows, stride = gridDim.y * kRows;
  if (im.b < 0 || first >= n_rows) return;   // padding

  const bool odd = C::OTHER && a.odd[u];   // (of whole units only)
  // Tiles before this item, of it and in total.
  int before = 0, Ti = 0, total = 0;
  if constexpr (C::kRowPlan) {
    before = a.ipre[item];
    Ti = a.ipre[item + 1] - before;
    total = a.ipre[a.n_items];
  } else {   // block reductions over items
    Ti = item_tiles<C>(a, item);
    for (int i = tid; i < a.n_items; i += kMergeWaves * kWave) {
      const int t = item_tiles<C>(a, i);
      total += t;
      if (i < item) before += t;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      before += __shfl_xor(before, off, kWave);
      total += __shfl_xor(total, off, kWave);
    }
    if (lane == 0) {
      red[0][w] = before;
      red[1][w] = total;
    }
    __syncthreads();
    before = total = 0;
#pragma unroll
    for (int k = 0; k < kMergeWaves; ++k) {
      before += red[0][k];
      total += red[1][k];
    }
  }
  int b0 = 0, b1 = -1;   // an empty context: zeros
  bool inside = false;   // the unit starts inside the first owner's range
  if (Ti > 0) {
    const int64_t N = (int64_t)units_per_item * total;
    const int64_t p = (int64_t)units_per_item * before + (int64_t)j * Ti;
    const int P = (int)min<int64_t>(a.n_blocks, N);   // as in the streaming kernel
    b0 = owner_of(p, N, P);
    inside = b0 * N / P < p;
    b1 = owner_of(p + Ti - 1, N, P);
    // one owner: written directly by the streaming kernel
    if (b0 == b1 && !odd) return;
  }

  const int D = C::OTHER ? a.head_dim : C::DP;
  const bool lane_out = !C::OTHER || 4 * lane < D;          // this lane writes outputs
  const bool lane_in = C::DP == 256 || lane < C::DP / 4;    // this lane holds partials
  const float vscale = C::FP8 ? a.v_scale[0] : 1.f;
  uint32_t om = 0;
  for (int n0 = first; n0 < n_rows; n0 += stride) {
    const int n = n0 + w / WPR;
    bool write = n < n_rows;
    const int rho = unit_row + n;   // row t * G + h of the request
    const int t = C::BLK ? rho / a.group : 0;
    const int qrow = im.qrow + t;
    const int hq = hk * a.group + rho - t * a.group;
    // The row's gate comes in under the partials' latency.
    u32x2 gv = {0u, 0u};
    if (write && a.gate && lane_out)
      gv = ld_g8(a.gate + (int64_t)qrow * a.gate_stride + (int64_t)hq * a.gate_hstride + 4 * lane);
    float m = -INFINITY, l = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (write && b0 != b1) {
      for (int bb = b0 + w % WPR; bb <= b1; bb += WPR * kMergeAhead) {
        f32x4 o[kMergeAhead];
        float2 ml[kMergeAhead];
#pragma unroll
        for (int k = 0; k < kMergeAhead; ++k) {
          const int bk = min(bb + WPR * k, b1);
          const int64_t slot = C::kRowPlan && a.by_owner
                                   ? 2 * (int64_t)bk + (inside && bk == b0 ? 1 : 0)
                                   : (int64_t)bk + u;
          const int64_t pr = slot * C::kRows + n;
          o[k] = reinterpret_cast<const f32x4*>(
              a.ws_o + pr * C::kRowFloats)[C::DP == 256 ? lane : lane & 31];
          ml[k] = reinterpret_cast<const float2*>(a.ws_ml)[pr];
        }
        float mn = m;
#pragma unroll
        for (int k = 0; k < kMergeAhead; ++k) {
          if (bb + WPR * k > b1) ml[k] = float2{-INFINITY, 0.f};   // a repeat of the last one
          mn = fmaxf(mn, ml[k].x);
        }
        // (NaN rows have a maximum of -inf and a NaN sum: the sum goes through)
        const float ref = mn == -INFINITY ? 0.f : mn;
        const float a1 = fast_exp2(m - ref);
        acc *= a1;
        l *= a1;
#pragma unroll
        for (int k = 0; k < kMergeAhead; ++k) {
          const float a2 = fast_exp2(ml[k].x - ref);
          if (bb + WPR * k <= b1) acc += o[k] * a2;
          l += ml[k].y * a2;
        }
        m = mn;
      }
    }
    if (WPR > 1) {
      __syncthreads();   // the previous rows are done with so / sm_m / sm_l
      so[w][lane] = acc;
      if (lane == 0) {
        sm_m[w] = m;
        sm_l[w] = l;
      }
      __syncthreads();
      if (w % WPR) write = false;   // the row's first wave goes on alone
      if (write) {
#pragma unroll
        for (int k = 1; k < WPR; ++k) {
          const float m2 = sm_m[w + k], l2 = sm_l[w + k];
          const float mn = fmaxf(m, m2);
          const float a1 = m == -INFINITY ? 0.f : fast_exp2(m - mn);
          const float a2 = m2 == -INFINITY ? 0.f : fast_exp2(m2 - mn);
          acc = acc * a1 + so[w + k][lane] * a2;
          l = l * a1 + l2 * a2;
          m = mn;
        }
      }
    }
    if constexpr (C::OTHER) {
      if (write && (b0 == b1 || __ballot(lane_in && not_finite(acc)))) {
        const int len = item_len(a, im);
        const int seen = C::BLK ? len - im.ext + t + 1 : len;
        const int row_bytes = C::FP8 ? D : 2 * D;
        RowState rs;
        attend_row<C::FP8>(
            rs, a.q + (int64_t)qrow * a.q_stride + (int64_t)hq * D,
            reinterpret_cast<uint32_t*>(&so[w][0]), D,
            a.rtt + clamp_i64(a.rpi[im.b], 0, a.rtt_rows - 1) * a.rtt_stride, 0, seen,
            a.pool_slots, a.seq_override > 0, a.k_pool + (int64_t)hk * row_bytes,
            a.v_pool + (int64_t)hk * row_bytes, (int64_t)a.hkv * row_bytes,
            a.scale_log2 * (C::FP8 ? a.k_scale[0] : 1.f), lane);
        om = max(om, write_row(rs, seen > 0 ? vscale / rs.l : 0.f, D,
                               a.out + (int64_t)qrow * a.out_stride + (int64_t)hq * D,
                               a.gate ? a.gate + (int64_t)qrow * a.gate_stride +
                                            (int64_t)hq * a.gate_hstride
                                      : nullptr,
                               lane));
        write = false;
      }
    }
    if (write) {
      // Lane (g, i) = (lane / kAcc, lane % kAcc) holds accumulator i of lane
      // group g (the partials' order); through LDS to dims 4 lane .. + 3.
      const float inv = l > 0.f || l != l ? vscale / l : 0.f;
      const int g = lane / C::kAcc, i = lane % C::kAcc;
      float* row_f = reinterpret_cast<float*>(&so[w][0]);
      wave_lds_sync();
      if (lane_in) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          row_f[C::FP8 ? 64 * g + 16 * r + i : 128 * (i >> 3) + 32 * g + 8 * r + (i & 7)] =
              acc[r] * inv;
      }
      wave_lds_sync();
      const f32x4 v = so[w][lane];
      u32x2 o = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      if (a.gate) {
        o[0] = gate_pair(o[0], gv[0]);
        o[1] = gate_pair(o[1], gv[1]);
      }
      if (lane_out) {
        om = max(om, max(o[0] & 0x7fffu, (o[0] >> 16) & 0x7fffu));
        om = max(om, max(o[1] & 0x7fffu, (o[1] >> 16) & 0x7fffu));
        *reinterpret_cast<u32x2*>(a.out + (int64_t)qrow * a.out_stride + (int64_t)hq * D +
                                  4 * lane) = o;
      }
    }
  }
  // One atomic per workgroup.
  if (!a.amax) return;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) om = max(om, (uint32_t)__shfl_xor((int)om, d, kWave));
  __syncthreads();
  if (lane == 0) red[0][w] = (int32_t)om;
  __syncthreads();
  if (w == 0) amax_commit(a.amax, lane < kMergeWaves ? (uint32_t)red[0][lane] : 0u);
}

}  // namespace

int make_decode_plan(int32_t n_items, int32_t num_q_heads, int32_t num_kv_heads,
                     int32_t head_dim, int32_t max_seq_len, int32_t num_workgroups,
                     DecodePlan* p) {
  (void)max_seq_len;
  if (n_items < 0) return fail(TF_ERR_INVALID, "decode: n_items=%d", n_items);
  if (n_items > kMaxItems)
    return fail(TF_ERR_UNSUPPORTED, "decode: %d requests in one call (at most %d)", n_items,
                kMaxItems);
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return fail(TF_ERR_INVALID, "decode: num_q_heads=%d not a multiple of num_kv_heads=%d",
                num_q_heads, num_kv_heads);
  if (num_workgroups < 0) return fail(TF_ERR_INVALID, "decode: num_workgroups=%d", num_workgroups);
  if (head_dim != kD) {
    // Other head dims run the one-wave-per-row kernel (attn_generic.hip)
    // here, which needs no workspace (tf_attn_rows takes one).
    if (!generic_head_dim(head_dim))
      return fail(TF_ERR_UNSUPPORTED,
                  "decode: head_dim=%d (a multiple of 8 between 8 and %d)", head_dim, kD);
    *p = DecodePlan{};
    p->generic = true;
    return TF_OK;
  }
  const int32_t group = num_q_heads / num_kv_heads;
  p->generic = false;
  // One persistent workgroup (4 waves) per CU measured fastest on MI355X.
  p->n_blocks = num_workgroups > 0 ? num_workgroups : device_cu_count();
  plan_units(n_items, num_kv_heads, (group + 15) / 16, 16, group < 16 ? group : 16, kD,
             false, p);
  return TF_OK;
}

void plan_units(int32_t n_items, int32_t num_kv_heads, int32_t n_hgroups, int32_t unit_rows,
                int32_t rows_used, int32_t row_floats, bool row_plan, DecodePlan* p) {
  p->n_hgroups = n_hgroups;
  p->rows_used = rows_used;
  p->n_units = (int64_t)n_items * num_kv_heads * n_hgroups;
  p->by_owner = row_plan && p->n_units > p->n_blocks;
  const int64_t slots = p->n_blocks + (p->by_owner ? p->n_blocks : p->n_units);
  const int64_t rows = slots * unit_rows;
  p->ml_bytes = (rows * 2 * 4 + 255) / 256 * 256;
  p->o_bytes = rows * row_floats * 4;
  p->total_bytes = p->ml_bytes + p->o_bytes;
  if (row_plan) p->total_bytes += 4 * (n_items + 1 + p->n_units);   // tile prefix, unit marks
}

}  // namespace tfa

namespace tfa {
namespace {

enum : int { kPhasePartial = 1, kPhaseMerge = 2 };

// The checks that every entry point of the streaming kernel shares.
int check_call(const char* fn, const void* q, int64_t q_row_stride, const void* k_pool,
               const void* v_pool, int64_t pool_slots, int32_t kv_dtype, const float* k_scale,
               const float* v_scale, const int64_t* req_to_token, int64_t rtt_rows,
               int64_t rtt_row_stride, int64_t rtt_cols, const int64_t* req_pool_indices,
               const int64_t* seq_lens, int32_t seq_len_override, int32_t num_q_heads,
               int32_t head_dim, const void* out, int64_t out_row_stride, const void* gate,
               int64_t gate_row_stride, int64_t gate_head_stride, const void* workspace,
               int64_t workspace_bytes, int64_t need_bytes) {
  if (kv_dtype != TF_DTYPE_BF16 && kv_dtype != TF_DTYPE_FP8_E4M3)
    return fail(TF_ERR_UNSUPPORTED, "%s: kv_dtype=%d", fn, kv_dtype);
  if (!q || !k_pool || !v_pool || !req_to_token || !req_pool_indices || !out)
    return fail(TF_ERR_INVALID, "%s: null pointer argument", fn);
  if (!seq_lens && seq_len_override <= 0)
    return fail(TF_ERR_INVALID, "%s: seq_lens is null and no override", fn);
  if (kv_dtype == TF_DTYPE_FP8_E4M3 && (!k_scale || !v_scale))
    return fail(TF_ERR_INVALID, "%s: fp8 pool needs k_scale and v_scale", fn);
  if (pool_slots < 1 || pool_slots > INT32_MAX || rtt_rows < 1 || rtt_cols < 1 ||
      rtt_row_stride < rtt_cols)
    return fail(TF_ERR_INVALID, "%s: bad pool/req_to_token extents", fn);
  if (!aligned16(q) || !aligned16(out) || !aligned16(k_pool) || !aligned16(v_pool) ||
      (q_row_stride * 2) % 16 || (out_row_stride * 2) % 16)
    return fail(TF_ERR_INVALID, "%s: q/out/pools must be 16-byte aligned", fn);
  if (q_row_stride < (int64_t)num_q_heads * head_dim ||
      out_row_stride < (int64_t)num_q_heads * head_dim)
    return fail(TF_ERR_INVALID, "%s: row stride smaller than num_q_heads*head_dim", fn);
  if (gate && (!aligned16(gate) || gate_row_stride % 8 || gate_head_stride % 8 ||
               gate_head_stride < head_dim))
    return fail(TF_ERR_INVALID, "%s: gate must be 16-byte aligned with strides of 8 elements", fn);
  if (need_bytes > 0 && (!workspace || workspace_bytes < need_bytes || !aligned16(workspace)))
    return fail(TF_ERR_INVALID, "%s: workspace needs %lld bytes, got %lld", fn,
                (long long)need_bytes, (long long)workspace_bytes);
  return TF_OK;
}

void set_args(DecodeArgs* a, const void* q, int64_t q_row_stride, const void* k_pool,
              const void* v_pool, int64_t pool_slots, const float* k_scale, const float* v_scale,
              const int64_t* req_to_token, int64_t rtt_rows, int64_t rtt_row_stride,
              int64_t rtt_cols, const int64_t* req_pool_indices, const int64_t* seq_lens,
              int32_t seq_len_override, int32_t n_items, int32_t num_q_heads,
              int32_t num_kv_heads, int32_t head_dim, float scale, void* out,
              int64_t out_row_stride, void* workspace, const void* gate, int64_t gate_row_stride,
              int64_t gate_head_stride, uint32_t* out_amax, const DecodePlan& p) {
  a->q = static_cast<const __bf16*>(q);
  a->q_stride = q_row_stride;
  a->k_pool = static_cast<const uint8_t*>(k_pool);
  a->v_pool = static_cast<const uint8_t*>(v_pool);
  a->pool_slots = pool_slots;
  a->k_scale = k_scale;
  a->v_scale = v_scale;
  a->rtt = req_to_token;
  a->rtt_rows = rtt_rows;
  a->rtt_stride = rtt_row_stride;
  a->rtt_cols = rtt_cols;
  a->rpi = req_pool_indices;
  a->seq_lens = seq_lens;
  a->seq_override = seq_len_override;
  a->n_items = n_items;
  a->hkv = num_kv_heads;
  a->group = num_q_heads / num_kv_heads;
  a->n_hg = p.n_hgroups;
  a->head_dim = head_dim;
  a->scale_log2 = scale * kLog2e;
  a->out = static_cast<__bf16*>(out);
  a->out_stride = out_row_stride;
  a->gate = static_cast<const __bf16*>(gate);
  a->gate_stride = gate_row_stride;
  a->gate_hstride = gate_head_stride;
  a->amax = out_amax;
  char* ws = static_cast<char*>(workspace);
  a->ws_ml = reinterpret_cast<float*>(ws);
  a->ws_o = reinterpret_cast<float*>(ws + p.ml_bytes);
  a->ipre = reinterpret_cast<int32_t*>(ws + p.ml_bytes + p.o_bytes);
  a->odd = a->ipre + n_items + 1;
  a->n_blocks = p.n_blocks;
  a->by_owner = p.by_owner;
}

// Launches the streaming kernel and / or the merge of one call.
template <class C>
int launch_rows(const DecodeArgs& a, const DecodePlan& p, int phases, hipStream_t s) {
  if (phases & kPhasePartial) {
    hipLaunchKernelGGL((decode_kernel<C>), dim3((unsigned)p.n_blocks), dim3(kWaves * kWave), 0, s,
                       a);
    const int rc = launch_status("tf_attn_decode partial launch");
    if (rc != TF_OK) return rc;
  }
  if (phases & kPhaseMerge) {
    // kWaves waves per (unit, head) row when the units average more than
    // three partials each, else one (measured: see decode_merge_kernel), and one
    // where that would be more than two workgroups per CU (86 requests on a grid
    // of 768, about three partials each: 11.2 us wide, 6.3 narrow).  With
    // many units most are not split: one workgroup per unit then, so that it
    // finds that out once.
    constexpr int kWideRows = kMergeWaves / kWaves;
    const bool wide = (int64_t)p.n_blocks > 2 * p.n_units &&
                      p.n_units * ((p.rows_used + kWideRows - 1) / kWideRows) <=
                          2 * device_cu_count();
    const int per_wg = wide ? kMergeWaves / kWaves : kMergeWaves;
    const bool many = p.n_units >= 2 * p.n_blocks;
    const dim3 grid((unsigned)p.n_units,
                    many ? 1u : (unsigned)((p.rows_used + per_wg - 1) / per_wg));
    const dim3 block(kMergeWaves * kWave);
    if (wide)
      hipLaunchKernelGGL((decode_merge_kernel<C, kWaves>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((decode_merge_kernel<C, 1>), grid, block, 0, s, a);
    return launch_status("tf_attn_decode merge launch");
  }
  return TF_OK;
}

int decode_launch(const void* q, int64_t q_row_stride, const void* k_pool, const void* v_pool,
                  int64_t pool_slots, int32_t kv_dtype, const float* k_scale,
                  const float* v_scale, const int64_t* req_to_token, int64_t rtt_rows,
                  int64_t rtt_row_stride, int64_t rtt_cols, const int64_t* req_pool_indices,
                  const int64_t* seq_lens, int32_t seq_len_override, const int32_t* items,
                  const int32_t* q_rows, int32_t n_items, int32_t num_q_heads,
                  int32_t num_kv_heads, int32_t head_dim, float scale, void* out,
                  int64_t out_row_stride, void* workspace, int64_t workspace_bytes,
                  int32_t max_seq_len, int32_t num_workgroups, const void* gate,
                  int64_t gate_row_stride, int64_t gate_head_stride, uint32_t* out_amax,
                  tf_stream_t stream, int phases) {
  clear_error();
  DecodePlan p;
  int rc = make_decode_plan(n_items, num_q_heads, num_kv_heads, head_dim, max_seq_len,
                            num_workgroups, &p);
  if (rc != TF_OK) return rc;
  if (n_items == 0) return TF_OK;
  rc = check_call("decode", q, q_row_stride, k_pool, v_pool, pool_slots, kv_dtype, k_scale,
                  v_scale, req_to_token, rtt_rows, rtt_row_stride, rtt_cols, req_pool_indices,
                  seq_lens, seq_len_override, num_q_heads, head_dim, out, out_row_stride, gate,
                  gate_row_stride, gate_head_stride, workspace, workspace_bytes, p.total_bytes);
  if (rc != TF_OK) return rc;
  if (p.n_units > INT32_MAX) return fail(TF_ERR_INVALID, "decode: too many units");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (p.generic) {   // head_dim != 256: everything happens in the "partial" phase
    if (!(phases & kPhasePartial)) return TF_OK;
    GenericAttnArgs g{};
    g.q = static_cast<const __bf16*>(q);
    g.q_stride = q_row_stride;
    g.k_pool = static_cast<const uint8_t*>(k_pool);
    g.v_pool = static_cast<const uint8_t*>(v_pool);
    g.pool_slots = pool_slots;
    g.fp8 = kv_dtype == TF_DTYPE_FP8_E4M3;
    g.k_scale = k_scale;
    g.v_scale = v_scale;
    g.rtt = req_to_token;
    g.rtt_rows = rtt_rows;
    g.rtt_stride = rtt_row_stride;
    g.rtt_cols = rtt_cols;
    g.rpi = req_pool_indices;
    g.seq_lens = seq_lens;
    g.seq_override = seq_len_override;
    g.items = items;
    g.q_rows = q_rows;
    g.work = nullptr;
    g.n_rows = n_items;
    g.hq = num_q_heads;
    g.hkv = num_kv_heads;
    g.head_dim = head_dim;
    g.scale_log2 = scale * kLog2e;
    g.out = static_cast<__bf16*>(out);
    g.out_stride = out_row_stride;
    g.gate = static_cast<const __bf16*>(gate);
    g.gate_stride = gate_row_stride;
    g.gate_hstride = gate_head_stride;
    g.amax = out_amax;
    return launch_generic_attn(g, s);
  }
  DecodeArgs a = {};
  a.items = items;
  a.q_rows = q_rows;
  set_args(&a, q, q_row_stride, k_pool, v_pool, pool_slots, k_scale, v_scale, req_to_token,
           rtt_rows, rtt_row_stride, rtt_cols, req_pool_indices, seq_lens, seq_len_override,
           n_items, num_q_heads, num_kv_heads, head_dim, scale, out, out_row_stride, workspace,
           gate, gate_row_stride, gate_head_stride, out_amax, p);
  if (kv_dtype == TF_DTYPE_FP8_E4M3)
    return launch_rows<Cfg<256, true, 1, false, false>>(a, p, phases, s);
  return launch_rows<Cfg<256, false, 1, false, false>>(a, p, phases, s);
}

// The kernel configuration of a tf_attn_rows call.
struct RowsPlan {
  DecodePlan p;
  int32_t groups;   // NG
  bool narrow;      // 128-dim tiles
};

int make_rows_plan(bool blocks, int32_t n_items, int32_t row_groups, int32_t num_q_heads,
                   int32_t num_kv_heads, int32_t head_dim, int32_t kv_dtype,
                   int32_t num_workgroups, RowsPlan* r) {
  if (n_items < 0 || num_workgroups < 0)
    return fail(TF_ERR_INVALID, "rows: n_items=%d num_workgroups=%d", n_items, num_workgroups);
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return fail(TF_ERR_INVALID, "rows: num_q_heads=%d not a multiple of num_kv_heads=%d",
                num_q_heads, num_kv_heads);
  const bool fp8 = kv_dtype == TF_DTYPE_FP8_E4M3;
  const bool narrow = head_dim <= 128 && !fp8;
  if (row_groups != 1 && (row_groups != 2 || !blocks))
    return fail(TF_ERR_INVALID, "rows: row_groups=%d (1, or 2 with blocks)", row_groups);
  if (blocks && head_dim != kD && row_groups != 2)
    return fail(TF_ERR_INVALID, "rows: row_groups=%d (2 at head dims other than %d)", row_groups,
                kD);
  if (head_dim != kD && (!generic_head_dim(head_dim) || (fp8 && head_dim % 16)))
    return fail(TF_ERR_UNSUPPORTED, "rows: head_dim=%d (a multiple of 8, for fp8 pools of 16, "
                "up to %d)", head_dim, kD);
  if (!blocks && n_items > kMaxItems)
    return fail(TF_ERR_UNSUPPORTED, "rows: %d requests in one call (at most %d)", n_items,
                kMaxItems);
  r->groups = row_groups;
  r->narrow = narrow;
  const int32_t rows = 16 * r->groups, group = num_q_heads / num_kv_heads;
  r->p = DecodePlan{};
  // One workgroup per CU, as for decode; two of the 128-dim ones, whose tiles
  // are half as large, fit and hide each other's latency (2 prompts of 100 to
  // 400 tokens beside 12 decodes, 32 / 8 heads of 128: 112 us with one of 64
  // rows per CU, 75 us with two of 32).
  r->p.n_blocks = num_workgroups > 0 ? num_workgroups : device_cu_count() * (narrow ? 2 : 1);
  plan_units(n_items < kMaxItems ? n_items : kMaxItems, num_kv_heads,
             blocks ? 1 : (group + rows - 1) / rows, rows, blocks || group > rows ? rows : group,
             r->narrow ? 128 : kD, blocks || head_dim != kD, &r->p);
  if (r->p.n_units > INT32_MAX) return fail(TF_ERR_INVALID, "rows: too many units");
  return TF_OK;
}

}  // namespace
}  // namespace tfa

extern "C" int64_t tf_attn_rows_workspace_bytes(int32_t has_blocks, int32_t n_items,
                                                int32_t row_groups, int32_t num_q_heads,
                                                int32_t num_kv_heads, int32_t head_dim,
                                                int32_t kv_dtype, int32_t num_workgroups) {
  using namespace tfa;
  clear_error();
  RowsPlan r;
  const int rc = make_rows_plan(has_blocks != 0, n_items, row_groups, num_q_heads, num_kv_heads,
                                head_dim, kv_dtype, num_workgroups, &r);
  return rc != TF_OK ? rc : r.p.total_bytes;
}

extern "C" int32_t tf_attn_rows(
    const void* q, int64_t q_row_stride, const void* k_pool, const void* v_pool,
    int64_t pool_slots, int32_t kv_dtype, const float* k_scale, const float* v_scale,
    const int64_t* req_to_token, int64_t rtt_rows, int64_t rtt_row_stride, int64_t rtt_cols,
    const int64_t* req_pool_indices, const int64_t* seq_lens, int32_t seq_len_override,
    const int32_t* blocks, int32_t n_items, int32_t row_groups, int32_t num_q_heads,
    int32_t num_kv_heads, int32_t head_dim, float scale, void* out, int64_t out_row_stride,
    void* workspace, int64_t workspace_bytes, int32_t num_workgroups, const void* gate,
    int64_t gate_row_stride, int64_t gate_head_stride, uint32_t* out_amax, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  RowsPlan r;
  int rc = make_rows_plan(blocks != nullptr, n_items, row_groups, num_q_heads, num_kv_heads,
                          head_dim, kv_dtype, num_workgroups, &r);
  if (rc != TF_OK) return rc;
  if (n_items == 0) return TF_OK;
  rc = check_call("rows", q, q_row_stride, k_pool, v_pool, pool_slots, kv_dtype, k_scale, v_scale,
                  req_to_token, rtt_rows, rtt_row_stride, rtt_cols, req_pool_indices, seq_lens,
                  seq_len_override, num_q_heads, head_dim, out, out_row_stride, gate,
                  gate_row_stride, gate_head_stride, workspace, workspace_bytes, r.p.total_bytes);
  if (rc != TF_OK) return rc;
  if (!aligned16(blocks)) return fail(TF_ERR_INVALID, "rows: blocks must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool fp8 = kv_dtype == TF_DTYPE_FP8_E4M3;
  // kMaxItems blocks per launch, one after the other in the same workspace.
  for (int32_t i0 = 0; i0 < n_items; i0 += kMaxItems) {
    const int32_t n = n_items - i0 < kMaxItems ? n_items - i0 : kMaxItems;
    RowsPlan part;
    rc = make_rows_plan(blocks != nullptr, n, row_groups, num_q_heads, num_kv_heads, head_dim,
                        kv_dtype, num_workgroups, &part);
    if (rc != TF_OK) return rc;
    DecodeArgs a = {};
    a.blocks = blocks ? reinterpret_cast<const RowItem*>(blocks) + i0 : nullptr;
    set_args(&a, q, q_row_stride, k_pool, v_pool, pool_slots, k_scale, v_scale, req_to_token,
             rtt_rows, rtt_row_stride, rtt_cols, req_pool_indices, seq_lens, seq_len_override, n,
             num_q_heads, num_kv_heads, head_dim, scale, out, out_row_stride, workspace, gate,
             gate_row_stride, gate_head_stride, out_amax, part.p);
    constexpr int kBoth = kPhasePartial | kPhaseMerge;
    const DecodePlan& p = part.p;
    if (part.narrow)
      rc = blocks ? launch_rows<Cfg<128, false, 2, true, true>>(a, p, kBoth, s)
                  : launch_rows<Cfg<128, false, 1, true, false>>(a, p, kBoth, s);
    else if (head_dim != kD && fp8)
      rc = blocks ? launch_rows<Cfg<256, true, 2, true, true>>(a, p, kBoth, s)
                  : launch_rows<Cfg<256, true, 1, true, false>>(a, p, kBoth, s);
    else if (head_dim != kD)
      rc = blocks ? launch_rows<Cfg<256, false, 2, true, true>>(a, p, kBoth, s)
                  : launch_rows<Cfg<256, false, 1, true, false>>(a, p, kBoth, s);
    else if (part.groups == 2 && fp8)
      rc = launch_rows<Cfg<256, true, 2, false, true>>(a, p, kBoth, s);
    else if (part.groups == 2)
      rc = launch_rows<Cfg<256, false, 2, false, true>>(a, p, kBoth, s);
    else if (fp8)
      rc = blocks ? launch_rows<Cfg<256, true, 1, false, true>>(a, p, kBoth, s)
                  : launch_rows<Cfg<256, true, 1, false, false>>(a, p, kBoth, s);
    else
      rc = blocks ? launch_rows<Cfg<256, false, 1, false, true>>(a, p, kBoth, s)
                  : launch_rows<Cfg<256, false, 1, false, false>>(a, p, kBoth, s);
    if (rc != TF_OK) return rc;
  }
  return TF_OK;
}

#define TF_DECODE_PARAMS                                                                    \
  const void *q, int64_t q_row_stride, const void *k_pool, const void *v_pool,            \
      int64_t pool_slots, int32_t kv_dtype, const float *k_scale, const float *v_scale,    \
      const int64_t *req_to_token, int64_t rtt_rows, int64_t rtt_row_stride,               \
      int64_t rtt_cols, const int64_t *req_pool_indices, const int64_t *seq_lens,          \
      int32_t seq_len_override, const int32_t *items, const int32_t *q_rows,               \
      int32_t n_items, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,        \
      float scale, void *out, int64_t out_row_stride, void *workspace,                     \
      int64_t workspace_bytes, int32_t max_seq_len, int32_t num_workgroups,                \
      const void *gate, int64_t gate_row_stride, int64_t gate_head_stride,                 \
      uint32_t *out_amax, tf_stream_t stream
#define TF_DECODE_ARGS                                                                      \
  q, q_row_stride, k_pool, v_pool, pool_slots, kv_dtype, k_scale, v_scale, req_to_token,   \
      rtt_rows, rtt_row_stride, rtt_cols, req_pool_indices, seq_lens, seq_len_override,    \
      items, q_rows, n_items, num_q_heads, num_kv_heads, head_dim, scale, out,             \
      out_row_stride, workspace, workspace_bytes, max_seq_len, num_workgroups, gate,       \
      gate_row_stride, gate_head_stride, out_amax, stream

extern "C" {

int64_t tf_attn_decode_workspace_bytes(int32_t n_items, int32_t num_q_heads,
                                       int32_t num_kv_heads, int32_t head_dim,
                                       int32_t max_seq_len, int32_t num_workgroups) {
  tfa::clear_error();
  tfa::DecodePlan p;
  const int rc = tfa::make_decode_plan(n_items, num_q_heads, num_kv_heads, head_dim,
                                       max_seq_len, num_workgroups, &p);
  if (rc != TF_OK) return rc;
  return p.total_bytes;
}

int32_t tf_attn_decode(TF_DECODE_PARAMS) {
  return tfa::decode_launch(TF_DECODE_ARGS, tfa::kPhasePartial | tfa::kPhaseMerge);
}

int32_t tf_attn_decode_partial(TF_DECODE_PARAMS) {
  return tfa::decode_launch(TF_DECODE_ARGS, tfa::kPhasePartial);
}

int32_t tf_attn_decode_merge(TF_DECODE_PARAMS) {
  return tfa::decode_launch(TF_DECODE_ARGS, tfa::kPhaseMerge);
}

}  // extern "C"

// ------------------------------------------------------------ no-allocation decode
// tf_attn_decode for callers that cannot allocate device memory: the split
// partials live in this library-owned array instead of a caller workspace.
// Every GPU the library runs on holds its own copy from module load until the
// process ends; all calls on one GPU share it (the partials need no
// initialisation: every one the merge reads was written earlier in the same
// call), so calls that overlap in time on one GPU race.
static constexpr int64_t kNoAllocScratchBytes = 32LL << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

namespace tfa {
namespace {

constexpr int kMaxDevices = 64;

// The device address of `scratch` on the current device, looked up once per
// device (the host-side name is only a handle for the lookup; passing it to a
// kernel would fault).
int noalloc_scratch(hipStream_t stream, void** ptr) {
  static std::mutex mu;
  static void* cache[kMaxDevices];
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(TF_ERR_HIP, "decode_noalloc: hipGetDevice: %s",
                                   hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(TF_ERR_UNSUPPORTED, "decode_noalloc: device %d", dev);
  if (stream) {
    hipDevice_t sdev = -1;
    e = hipStreamGetDevice(stream, &sdev);
    if (e != hipSuccess)
      return fail(TF_ERR_HIP, "decode_noalloc: hipStreamGetDevice: %s", hipGetErrorString(e));
    if (sdev != dev)
      return fail(TF_ERR_INVALID, "decode_noalloc: the stream is on device %d, device %d is "
                  "current (make the stream's device current)", (int)sdev, dev);
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!cache[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(TF_ERR_HIP, "decode_noalloc: hipGetSymbolAddress(scratch): %s",
                  hipGetErrorString(e));
    cache[dev] = p;
  }
  *ptr = cache[dev];
  return TF_OK;
}

}  // namespace
}  // namespace tfa

extern "C" int32_t tf_attn_decode_noalloc(
    const void* q, int64_t q_row_stride, const void* k_pool, const void* v_pool,
    int64_t pool_slots, int32_t kv_dtype, const float* k_scale, const float* v_scale,
    const int64_t* req_to_token, int64_t rtt_rows, int64_t rtt_row_stride, int64_t rtt_cols,
    const int64_t* req_pool_indices, const int64_t* seq_lens, int32_t seq_len_override,
    const int32_t* items, const int32_t* q_rows, int32_t n_items, int32_t num_q_heads,
    int32_t num_kv_heads, int32_t head_dim, float scale, void* out, int64_t out_row_stride,
    int32_t max_seq_len, int32_t num_workgroups, const void* gate, int64_t gate_row_stride,
    int64_t gate_head_stride, uint32_t* out_amax, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  DecodePlan p;
  const int rc = make_decode_plan(n_items, num_q_heads, num_kv_heads, head_dim, max_seq_len,
                                  num_workgroups, &p);
  if (rc != TF_OK) return rc;
  if (p.total_bytes > kNoAllocScratchBytes)
    return fail(TF_ERR_UNSUPPORTED,
                "decode_noalloc: this call needs %lld bytes of split scratch, the static buffer "
                "holds %lld (fewer requests or workgroups per call, or tf_attn_decode with a "
                "workspace)", (long long)p.total_bytes, (long long)kNoAllocScratchBytes);
  void* ws = nullptr;
  const int rc2 = noalloc_scratch(reinterpret_cast<hipStream_t>(stream), &ws);
  if (rc2 != TF_OK) return rc2;
  void* workspace = ws;
  const int64_t workspace_bytes = kNoAllocScratchBytes;
  return decode_launch(TF_DECODE_ARGS, kPhasePartial | kPhaseMerge);
}
