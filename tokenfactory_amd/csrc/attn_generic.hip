// Slot attention for head dims other than 256, one wave per query row: decode and
// extend rows of any head_dim that is a multiple of 8, up to 256.
// tf_attn_decode / tf_attn_extend, which take no workspace at these head dims,
// route here; so do fp8 pools whose head dim is not a multiple of 16.
// tf_attn_rows (decode.hip) runs everything else on MFMAs.
//
// Same semantics as those kernels (qwen3_8/full_attention.py:163-283): row
// (token t, q head h) of request b attends to context positions 0 .. P + t,
// P = L_b - ext_b, q head h reads kv head h / G, slot ids come from
// req_to_token (negative ids index from the pool's end in a bsz == 1 call,
// then every id is clamped into the pool), fp8-e4m3 pools are read with their
// per-tensor scales, and the optional output gate is applied to the rounded
// output as bf16(bf16(o) * bf16(silu(g))).
//
// One wave per query row.  Keys go 64 at a time: lane j scores key k0 + j
// against the whole q row (held by every lane as packed bf16), the wave takes
// the tile's max and sum, and each lane accumulates two output dims (2l, 2l + 1,
// and 128 + 2l, 129 + 2l for head_dim > 128) over the tile's keys in fp32.
#include <math.h>

#include "attn_row.h"
#include "tf_common.h"
#include "tf_internal.h"

namespace tfa {

namespace {

constexpr int kGenWaves = 4;
constexpr int kGenThreads = kGenWaves * kWave;

template <bool FP8>
__global__ void __launch_bounds__(kGenThreads) generic_attn_kernel(GenericAttnArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t wid = (int64_t)blockIdx.x * kGenWaves + threadIdx.x / kWave;
  const int G = a.hq / a.hkv;
  const int D = a.head_dim;

  // This wave's query row.
  int b, h, hk;
  int64_t qrow, limit, L;
  if (a.work) {   // extend: work entry wid / 256, row (wid % 256) of it
    const int64_t e = wid / kExtendItemRows;
    if (e >= a.n_rows) return;
    const int32_t* wk = a.work + 8 * e;
    const int ext = wk[4];
    if (ext <= 0) return;                      // padding entry of a device-built list
    const int r = wk[2] + (int)(wid % kExtendItemRows);
    if (r >= ext * G) return;
    b = wk[0];
    hk = wk[1];
    const int t = r / G;
    h = hk * G + r % G;
    qrow = (int64_t)wk[3] + t;
    L = a.seq_override > 0 ? (int64_t)a.seq_override : a.seq_lens[b];
    if (L > a.rtt_cols) L = a.rtt_cols;
    limit = L - ext + t;                       // last visible key
  } else {        // decode: item wid / hq, head wid % hq
    const int64_t i = wid / a.hq;
    if (i >= a.n_rows) return;
    b = a.items ? a.items[i] : (int)i;
    if (b < 0) return;                         // padding item
    qrow = a.q_rows ? a.q_rows[i] : b;
    h = (int)(wid % a.hq);
    hk = h / G;
    L = a.seq_override > 0 ? (int64_t)a.seq_override : a.seq_lens[b];
    if (L > a.rtt_cols) L = a.rtt_cols;
    limit = L - 1;
  }
  // A row with no visible key (a decode item with seq_len 0, an extend row
  // past a too-short context) is all zeros, as the reference's fully masked
  // scaled_dot_product_attention returns it and as the tuned kernels write it.
  const int64_t nkeys = limit + 1;

  const int64_t rrow = clamp_i64(a.rpi[b], 0, a.rtt_rows - 1);
  const int64_t* rtt = a.rtt + rrow * a.rtt_stride;
  const bool wrap = a.seq_override > 0;
  const int esz = FP8 ? 1 : 2;
  const int64_t row_bytes = (int64_t)a.hkv * D * esz;
  const uint8_t* kbase = a.k_pool + (int64_t)hk * D * esz;
  const uint8_t* vbase = a.v_pool + (int64_t)hk * D * esz;

  __shared__ uint32_t qs[kGenWaves][kRowMaxD / 2];
  RowState st;
  attend_row<FP8>(st, a.q + qrow * a.q_stride + (int64_t)h * D, qs[threadIdx.x / kWave], D, rtt, 0,
                  nkeys, a.pool_slots, wrap, kbase, vbase, row_bytes,
                  a.scale_log2 * (FP8 ? a.k_scale[0] : 1.f), lane);
  const float inv = nkeys > 0 ? (FP8 ? a.v_scale[0] : 1.f) / st.l : 0.f;
  amax_commit(a.amax, write_row(st, inv, D, a.out + qrow * a.out_stride + (int64_t)h * D,
                                a.gate ? a.gate + qrow * a.gate_stride +
                                             (int64_t)h * a.gate_hstride
                                       : nullptr,
                                lane));
}

}  // namespace

bool generic_head_dim(int32_t head_dim) {
  return head_dim != 256 && head_dim >= 8 && head_dim <= kRowMaxD && head_dim % 8 == 0;
}

int launch_generic_attn(const GenericAttnArgs& a, hipStream_t stream) {
  const int64_t waves = a.work ? (int64_t)a.n_rows * kExtendItemRows : (int64_t)a.n_rows * a.hq;
  const int64_t blocks = (waves + kGenWaves - 1) / kGenWaves;
  if (blocks <= 0) return TF_OK;
  if (blocks > INT32_MAX) return fail(TF_ERR_INVALID, "attention: too many rows");
  if (a.fp8)
    hipLaunchKernelGGL(generic_attn_kernel<true>, dim3((unsigned)blocks), dim3(kGenThreads), 0,
                       stream, a);
  else
    hipLaunchKernelGGL(generic_attn_kernel<false>, dim3((unsigned)blocks), dim3(kGenThreads), 0,
                       stream, a);
  return launch_status("generic attention launch");
}

}  // namespace tfa
