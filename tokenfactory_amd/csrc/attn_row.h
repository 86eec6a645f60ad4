// One query row's attention by one wave, fp32 throughout: the whole of
// attn_generic.hip's work, and the streaming kernel's second look at rows whose
// accumulators do not stay finite (decode.hip).
//
// Online softmax over a run of 64 keys at a time, one key per lane for the
// scores; O holds dims 2 lane, 2 lane + 1, 128 + 2 lane, 129 + 2 lane.  Only what
// the row sees is read.
#pragma once

#include "tf_common.h"

namespace tfa {

constexpr int kRowMaxD = 256;

struct RowState {
  float m = -INFINITY, l = 0.f;   // max (log2 units) and sum of 2^(s - m)
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, kWave));
  return v;
}

// 8 elements of a K or V row (bf16, or e4m3 when FP8) at element offset e.
template <bool FP8>
__device__ __forceinline__ void load8(const uint8_t* row, int e, float (&x)[8]) {
  if (FP8) {
    const u32x2 r = *reinterpret_cast<const u32x2*>(row + e);
    const u32x4 b = e4m3x8_to_bf16x8(r[0], r[1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(b[i] << 16);
      x[2 * i + 1] = __uint_as_float(b[i] & 0xffff0000u);
    }
  } else {
    const u32x4 r = *reinterpret_cast<const u32x4*>(row + 2 * e);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(r[i] << 16);
      x[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
}

// Two consecutive elements of a row at element offset e (e even).
template <bool FP8>
__device__ __forceinline__ void load2(const uint8_t* row, int e, float& x0, float& x1) {
  if (FP8) {
    const uint32_t b = e4m3x2_to_bf16x2<false>(*reinterpret_cast<const uint16_t*>(row + e));
    x0 = __uint_as_float(b << 16);
    x1 = __uint_as_float(b & 0xffff0000u);
  } else {
    const uint32_t r = *reinterpret_cast<const uint32_t*>(row + 2 * e);
    x0 = __uint_as_float(r << 16);
    x1 = __uint_as_float(r & 0xffff0000u);
  }
}

// The row qp (bf16 [D]) over keys [k0, k1) of rtt, into st.  q: kRowMaxD / 2
// dwords of LDS of this wave's own (every lane reads the same word: a broadcast;
// wave_lds_sync orders every lane's writes before any lane's reads).
template <bool FP8>
__device__ __forceinline__ void attend_row(RowState& st, const __bf16* qp, uint32_t* q, int D,
                                           const int64_t* rtt, int64_t k0, int64_t k1,
                                           int64_t pool_slots, bool wrap, const uint8_t* kbase,
                                           const uint8_t* vbase, int64_t row_bytes, float sl2,
                                           int lane) {
  wave_lds_sync();   // the row before is done with q
  for (int i = lane; i < D / 2; i += kWave) q[i] = reinterpret_cast<const uint32_t*>(qp)[i];
  wave_lds_sync();
  const int d0 = 2 * lane, d1 = 128 + 2 * lane;
  for (; k0 < k1; k0 += kWave) {
    const int64_t k = k0 + lane;
    const bool live = k < k1;
    const int64_t slot = live ? pool_row(rtt[k], pool_slots, wrap) : 0;
    float s = -INFINITY;
    if (live) {
      const uint8_t* kr = kbase + slot * row_bytes;
      float dot = 0.f;
      for (int e = 0; e < D; e += 8) {
        float x[8];
        load8<FP8>(kr, e, x);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t qq = q[(e >> 1) + i];
          dot = fmaf(__uint_as_float(qq << 16), x[2 * i], dot);
          dot = fmaf(__uint_as_float(qq & 0xffff0000u), x[2 * i + 1], dot);
        }
      }
      s = dot * sl2;
    }
    const float mt = wave_max(s);
    const float mnew = fmaxf(st.m, mt);        // finite: key k0 is live
    const float alpha = exp2f(st.m - mnew);
    const float p = live ? exp2f(s - mnew) : 0.f;
    st.l = st.l * alpha + wave_sum(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) st.acc[i] *= alpha;
    st.m = mnew;
    const int n = (int)min<int64_t>(kWave, k1 - k0);
    for (int j = 0; j < n; ++j) {
      const float pj = __shfl(p, j, kWave);
      const int64_t sj = __shfl(slot, j, kWave);
      const uint8_t* vr = vbase + sj * row_bytes;
      if (d0 < D) {
        float x0, x1;
        load2<FP8>(vr, d0, x0, x1);
        st.acc[0] = fmaf(pj, x0, st.acc[0]);
        st.acc[1] = fmaf(pj, x1, st.acc[1]);
      }
      if (d1 < D) {
        float x0, x1;
        load2<FP8>(vr, d1, x0, x1);
        st.acc[2] = fmaf(pj, x0, st.acc[2]);
        st.acc[3] = fmaf(pj, x1, st.acc[3]);
      }
    }
  }
}

// The row's outputs acc * inv, gated where grow is not NULL; returns the largest
// |value| written (bf16 bits).
__device__ __forceinline__ uint32_t write_row(const RowState& st, float inv, int D, __bf16* orow,
                                              const __bf16* grow, int lane) {
  uint32_t omax = 0;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int d = 128 * u + 2 * lane;
    if (d >= D) continue;
    uint32_t o = pack_bf16(st.acc[2 * u] * inv, st.acc[2 * u + 1] * inv);
    if (grow) o = gate_pair(o, *reinterpret_cast<const uint32_t*>(grow + d));
    omax = max(omax, max(o & 0x7fffu, (o >> 16) & 0x7fffu));
    *reinterpret_cast<uint32_t*>(orow + d) = o;
  }
  return omax;
}

}  // namespace tfa
