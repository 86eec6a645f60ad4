// Two narrow bf16 linears of one input: the per-head gate projections in_proj_b
// and in_proj_a of the linear-attention layers (qwen3_8/linear_attention.py:
// 311-314; 48 output columns each at hidden 5120), bf16(x w^T) with fp32
// accumulation, optionally with max |x| per row block for the FP8 quantisation
// of the same x (fp8_triton.py:128).
//
// Bound by latency at decode sizes and by L2 reads of x and the weights above: a
// workgroup owns MT 16-row and NT 16-column tiles and its sixteen waves split K,
// with kUnroll 32-wide steps of loads in flight each; the operands go from memory
// straight to v_mfma_f32_16x16x32_bf16 (no LDS staging: nothing is reused inside
// a wave), and the waves' partial sums meet in LDS.  All columns in one workgroup
// (x read once) was 37 us at 8 rows and 40 at 1900.
// Measured at hidden 5120, 48 + 48 columns, against one library product per
// weight and a separate max |x| pass: 48 rows 12 us (2 x 15.7 + 4), 1900 rows
// 24 us (2 x 15 + 7).  What is left at decode is the misses of few CUs: a split of
// K over workgroups would need a second launch for the sums.
#include "tf_common.h"
#include "tf_internal.h"

namespace tfa {
namespace {

constexpr int kWaves = 16;
constexpr int kThreads = kWaves * kWave;
constexpr int kStep = 32;      // K per MFMA
constexpr int kUnroll = 5;     // steps with their loads in flight (10: no faster)
constexpr int kMaxCols = 64;   // per weight

struct NarrowArgs {
  const __bf16* x;
  int64_t xs;
  int32_t rows, steps, n;      // steps: K / 32; n: columns per weight
  const __bf16* w[2];          // [n, K]
  uint16_t* out[2];            // bf16 [rows, n], row stride os
  int64_t os;
  uint32_t* amax;              // optional: max |x| bits per row block
};

// Workgroup (x, y): row tiles MT x .., column tiles NT (y % colblocks) .. of
// weight y / colblocks.
template <int NT, int MT>
__global__ void __launch_bounds__(kThreads) narrow_kernel(NarrowArgs a) {
  __shared__ f32x4 part[kWaves][MT * NT][kWave];
  __shared__ uint32_t red[kWaves];
  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int g = lane >> 4, r = lane & 15;
  const int row0 = blockIdx.x * 16 * MT;
  const int half = gridDim.y / 2;
  const int which = blockIdx.y >= half ? 1 : 0;
  const int col0 = (blockIdx.y - which * half) * 16 * NT;
  const int64_t K = (int64_t)a.steps * kStep;

  const __bf16* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)   // rows and columns past the end repeat the last one
    xp[m] = a.x + (int64_t)min(row0 + 16 * m + r, a.rows - 1) * a.xs + 8 * g;
  const __bf16* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    wp[t] = a.w[which] + (int64_t)min(col0 + 16 * t + r, a.n - 1) * K + 8 * g;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t mx = 0;
  const int s0 = a.steps * w / kWaves, s1 = a.steps * (w + 1) / kWaves;
  auto load = [&](int s, u32x4 (&xv)[MT], u32x4 (&wv)[NT]) {
    const int64_t k = (int64_t)kStep * s;
#pragma unroll
    for (int m = 0; m < MT; ++m) xv[m] = ld_g16(xp[m] + k);
#pragma unroll
    for (int t = 0; t < NT; ++t) wv[t] = ld_g16(wp[t] + k);
  };
  auto step = [&](const u32x4 (&xv)[MT], const u32x4 (&wv)[NT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      mx = max(mx, abs_max8(xv[m]));
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[m][t] = mfma_16x16x32(xv[m], wv[t], acc[m][t]);
    }
  };
  int s = s0;
  for (; s + kUnroll <= s1; s += kUnroll) {
    u32x4 xv[kUnroll][MT], wv[kUnroll][NT];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) load(s + u, xv[u], wv[u]);
    __builtin_amdgcn_sched_barrier(0);   // all loads in flight before the first product
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) step(xv[u], wv[u]);
  }
  for (; s < s1; ++s) {
    u32x4 xv[MT], wv[NT];
    load(s, xv, wv);
    step(xv, wv);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) part[w][m * NT + t][lane] = acc[m][t];
  const bool want_max = a.amax != nullptr && blockIdx.y == 0;
  if (want_max) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, d, kWave));
    if (lane == 0) red[w] = mx;
  }
  __syncthreads();
  if (want_max && threadIdx.x == 0) {
#pragma unroll
    for (int k = 1; k < kWaves; ++k) mx = max(mx, red[k]);
    a.amax[blockIdx.x] = mx;
  }
  // Tile i: lane (g, r) holds rows 4 g .. + 3 of column r.
  for (int i = w; i < MT * NT; i += kWaves) {
    f32x4 v = part[0][i][lane];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) v += part[k][i][lane];
    const int m = i / NT, t = i - m * NT;
    const int col = col0 + 16 * t + r;
    uint16_t* o = a.out[which];
    if (col >= a.n) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = row0 + 16 * m + 4 * g + e;
      if (row < a.rows) o[(int64_t)row * a.os + col] = (uint16_t)(pack_bf16(v[e], 0.f) & 0xffffu);
    }
  }
}

// Two row tiles and two column tiles per workgroup (half the L2 reads: 1900 rows
// 24 us) once a quarter of the CUs still have a row block, one of each below,
// where the CUs' outstanding misses bound it.
int narrow_rows(int64_t rows) { return rows > 16LL * device_cu_count() / 4 ? 32 : 16; }

}  // namespace
}  // namespace tfa

extern "C" {

int32_t tf_narrow_linear2_blocks(int64_t rows) {
  tfa::clear_error();
  if (rows < 0 || rows > INT32_MAX / 2)
    return tfa::fail(TF_ERR_INVALID, "narrow_linear2_blocks: rows=%lld", (long long)rows);
  const int per = tfa::narrow_rows(rows);
  return (int32_t)((rows + per - 1) / per);
}

int32_t tf_narrow_linear2(const void* x, int64_t x_row_stride, int64_t rows, int64_t k,
                          const void* w0, const void* w1, int32_t n, void* out0, void* out1,
                          int64_t out_row_stride, uint32_t* amax_partials, tf_stream_t stream) {
  using namespace tfa;
  clear_error();
  if (rows < 0 || rows > INT32_MAX / 2 || k <= 0 || k % kStep || k > INT32_MAX / 2)
    return fail(TF_ERR_INVALID, "narrow_linear2: rows=%lld k=%lld (a multiple of %d)",
                (long long)rows, (long long)k, kStep);
  if (n <= 0 || n > kMaxCols)
    return fail(TF_ERR_UNSUPPORTED, "narrow_linear2: n=%d (1 to %d)", n, kMaxCols);
  if (x_row_stride < k || x_row_stride % 8 || out_row_stride < n)
    return fail(TF_ERR_INVALID, "narrow_linear2: strides %lld / %lld (x rows 16-byte multiples)",
                (long long)x_row_stride, (long long)out_row_stride);
  if (rows == 0) return TF_OK;
  if (!x || !w0 || !w1 || !out0 || !out1)
    return fail(TF_ERR_INVALID, "narrow_linear2: null pointer");
  if (!aligned16(x) || !aligned16(w0) || !aligned16(w1) ||
      (reinterpret_cast<uintptr_t>(out0) & 1u) || (reinterpret_cast<uintptr_t>(out1) & 1u) ||
      (reinterpret_cast<uintptr_t>(amax_partials) & 3u))
    return fail(TF_ERR_INVALID, "narrow_linear2: x and the weights must be 16-byte aligned");
  NarrowArgs a;
  a.x = static_cast<const __bf16*>(x);
  a.xs = x_row_stride;
  a.rows = (int32_t)rows;
  a.steps = (int32_t)(k / kStep);
  a.n = n;
  a.w[0] = static_cast<const __bf16*>(w0);
  a.w[1] = static_cast<const __bf16*>(w1);
  a.out[0] = static_cast<uint16_t*>(out0);
  a.out[1] = static_cast<uint16_t*>(out1);
  a.os = out_row_stride;
  a.amax = amax_partials;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int per = narrow_rows(rows);
  const dim3 grid((unsigned)((rows + per - 1) / per), (unsigned)(2 * ((n + per - 1) / per)));
  if (per == 32)
    hipLaunchKernelGGL((narrow_kernel<2, 2>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((narrow_kernel<1, 1>), grid, dim3(kThreads), 0, s, a);
  return launch_status("tf_narrow_linear2 launch");
}

}  // extern "C"
