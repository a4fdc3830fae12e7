// What the two kernels of the fp32 scan of small states share (ssd_f32.hip, ssd_f32_long.hip): arguments, sums that keep what they lose, a chunk token by token.
#pragma once
#include "ssd_common.hpp"

namespace ssdk {

constexpr int FQ = 64, FN = 16;       // tokens a chunk (their steps are a wave's lanes), d_state

struct F3Args {
  const float *x, *dt, *Bm, *Cm, *A, *D, *dt_bias, *init;
  float *y, *final_state, *total_decay;
  int L, H, P, G, hpg, nch;
  int two, split, len0, len1, plen, npre;        // ssd_f32.hip
  float *loc, *segdec;                           // ssd_f32_long.hip: [segment][batch][head][P][16] local states, [segment][batch][head] sums of dt A
  int nseg, seg_chunks;
  int64_t xsb, xsl, dsb, dsl, bsb, bsl, bsg, csb, csl, csg, ysb, ysl;
  int softplus, group_map;
  float dt_min, dt_max;
};

__device__ __forceinline__ float rdlane(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ __forceinline__ float from_lane(float v, int l) { return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * l, __float_as_int(v))); }
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// a step of inclusive sums over lanes as value + what its rounding lost
template <int CTRL, int ROWMASK>
__device__ __forceinline__ void scan_step(float& hi, float& lo) {
  const float b = dpp_shift<CTRL, ROWMASK>(hi), bl = dpp_shift<CTRL, ROWMASK>(lo);
  const float s = hi + b, bb = s - hi;
  lo = (lo + bl) + ((hi - (s - bb)) + (b - bb));
  hi = s;
}
template <bool FINE> __device__ __forceinline__ float exp_of(float v) { return FINE ? expf(v) : __expf(v); }

// A chunk token by token, as the recurrence has it (ssd_generic.hip): S, y of the wave's columns; d and da are of token `lane`.  Returns the sum of da.
template <bool OUT>
__device__ __forceinline__ float march(const F3Args& a, const float* xb, const float* Bb, const float* Cb, int t0, int tt, float d, float da, float Dh, int lc, int q, int b, int h,
                                       int pt, f32x4& S) {
  float sum = 0.f;
#pragma unroll 1
  for (int t1 = 0; t1 < tt; t1 += 4) {
    float x[4];
    f32x4 B[4], C[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t t = t0 + min(t1 + j, tt - 1);
      x[j] = xb[t * a.xsl + lc];
      B[j] = *(const f32x4*)(Bb + t * a.bsl + 4 * q);
      if constexpr (OUT) C[j] = *(const f32x4*)(Cb + t * a.csl + 4 * q);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (t1 + j >= tt) break;
      const float dat = rdlane(da, t1 + j), dec = expf(dat), xv = rdlane(d, t1 + j) * x[j];
      float acc = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        S[r] = fmaf(dec, S[r], xv * B[j][r]);
        if constexpr (OUT) acc = fmaf(S[r], C[j][r], acc);
      }
      sum += dat;
      if constexpr (OUT) {
        acc += __shfl_xor(acc, 32, 64);
        acc += __shfl_xor(acc, 16, 64);
        if (q == 0) a.y[(int64_t)b * a.ysb + (int64_t)(t0 + t1 + j) * a.ysl + (int64_t)h * a.P + 16 * pt + lc] = fmaf(Dh, x[j], acc);
      }
    }
  }
  return sum;
}

}  // namespace ssdk
