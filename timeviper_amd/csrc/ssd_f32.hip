// S3 (fp32, d_state 16, head_dim a multiple of 16): the chunked scan of ssd_chunked.hip on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 products
// and sums, 4 columns of contraction a step).
//
// ssd_chunked.hip's work-groups were LDS reads: an operand a fused multiply-add from LDS, x and M through it, y written, read back and written again.  Here a WAVE takes
// 16 columns of a head through a segment of chunks of 64 tokens, and nothing but the tokens' decays passes LDS, because the operands chain:
//   * G^T = B C^T puts, in a lane, four source tokens of one output token (rows 4 (lane / 16) + r, column lane % 16); numbering the four steps of a
//     contraction of 16 tokens the same way (step r, quarter q: token 4 q + r), M^T = decays x dt x G^T is the operand of Y^T += x^T M^T as it leaves G;
//   * the state S^T += (w B)^T x leaves, in a lane, four entries n of one column p: the operand of Y^T = S C^T as it is, and 16-byte rows in memory;
//   * Y^T leaves four neighbouring columns of one token: 16-byte stores.
// Two launches: the state that every segment but the last leaves from a zero start; then a segment folds its predecessors' (in order, as the recurrence) and
// marches, writing y once.  How long a segment is: chunks_a_segment; the fold reads 1 KB a predecessor and wave.
// Products for a wave and chunk: 40 for G (again by each of a head's P / 16 waves), 40 + 16 for Y, 16 for S, 32 cycles each.
// Measured (32 heads x 64, 2 groups; ssd_chunked.hip's kernels -> here): 1 024 tokens 38 -> 21 us, 4 096: 128 -> 52, 2 x 4 096: 226 -> 91,
// 2 x 128: 23 -> 13.  Error of the final state against 64 bits 1.3e-7 (5e-7 .. 3e-6 with weights of differences of sums), of y 1.6e-7 (1.9e-7).
#include "ssd_common.hpp"

namespace {
using namespace ssdk;

constexpr int FQ = 64, FN = 16;       // tokens a chunk, d_state

struct F3Args {
  const float *x, *dt, *Bm, *Cm, *A, *D, *dt_bias, *init;
  float *y, *final_state, *total_decay;
  float *loc, *segdec;                // [segment][batch][head][P][16] local states, [segment][batch][head] sums of dt A
  int L, H, P, G, nch, nseg, seg_chunks;
  int64_t xsb, xsl, dsb, dsl, bsb, bsl, bsg, csb, csl, csg, ysb, ysl;
  int softplus, group_map;
  float dt_min, dt_max;
};

__device__ __forceinline__ float rdlane(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ __forceinline__ float from_lane(float v, int l) { return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * l, __float_as_int(v))); }
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// inclusive sums over the lanes as value + what its rounding lost (an infinite sum has lost nothing)
template <int CTRL, int ROWMASK>
__device__ __forceinline__ void scan_step(float& hi, float& lo) {
  const float b = dpp_shift<CTRL, ROWMASK>(hi), bl = dpp_shift<CTRL, ROWMASK>(lo);
  const float s = hi + b, bb = s - hi;
  lo = (lo + bl) + ((hi - (s - bb)) + (b - bb));
  hi = s;
}
__device__ __forceinline__ float scan_both(float v, float& lost) {
  lost = 0.f;
  scan_step<0x111, 0xf>(v, lost);   // row_shr:1
  scan_step<0x112, 0xf>(v, lost);   // row_shr:2
  scan_step<0x114, 0xf>(v, lost);   // row_shr:4
  scan_step<0x118, 0xf>(v, lost);   // row_shr:8
  scan_step<0x142, 0xa>(v, lost);   // row_bcast:15 -> rows 1, 3
  scan_step<0x143, 0xc>(v, lost);   // row_bcast:31 -> rows 2, 3
  lost = fabsf(v) < INFINITY ? lost : 0.f;
  return v;
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

// OUT: the second launch.  FINE: for the lengths that the token recurrence had before (48 - 64 tokens, more than 4 096), whose error and whose results at extreme steps are kept:
//   * two tokens' decay is the difference of their sums AND of what these have lost (a sum over a chunk is rounded by its own size, not by the difference's);
//   * the four steps of a contraction of 16 tokens are numbered in time (step r, quarter q: token 4 r + q; the rows of G^T are dealt out to match), so that what weighs most is added
//     last and rounded once, as by the recurrence; B has dt, and its sum with C over n is a tree;
//   * the decays of the state's weights are sums that keep what they lose, and their exponentials are the recurrence's own;
//   * a chunk with a token that leaves nothing of what was before it (dt A below -80, an infinite dt among them), or whose dt or dt A is otherwise out of the ordinary, goes token by
//     token (dt B, sums of dt A and differences of them are infinite or NaN there while the recurrence's products are not).
// Error against 64 bits, recurrence | here, 64 tokens of 32 heads x 64 that decay by e^-52: y 7.5e-8 | 7.2e-8, state 6.0e-8 | 5.7e-8; by e^-15: 8.8e-8 | 8.6e-8, 7.0e-8 | 6.7e-8; slowly:
// 2.2e-7 | 1.4e-7, 2.8e-7 | 1.6e-7; 5 000 tokens: 7.3e-8 | 6.9e-8, 6.1e-8 | 5.5e-8, slowly 4.0e-6 | 3.7e-7 (steps numbered as at the other lengths: 8.4e-8 for the first).
// All of this takes 5 - 12 % (64 tokens 7.8 -> 8.8 us, 8 192: 95 -> 99.5): the lengths between are as they were.  A reset in every chunk: 64 tokens 21 us (token by token
// 24), 8 192: 269 (2 695).
template <bool OUT, bool FINE>
__global__ __launch_bounds__(256) void ssd_f32_kernel(F3Args a) {
  __shared__ __attribute__((aligned(16))) float sv[4][FINE ? 4 : 3][FQ];         // a wave's own: cs, dt, weights of the state, what cs has lost
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, q = lane >> 4;
  auto tok = [&](int r) __attribute__((always_inline)) { return FINE ? 4 * r + q : 4 * q + r; };       // of the 16: step r's token in this quarter
  const int row = FINE ? (lc & 3) << 2 | lc >> 2 : lc, slot = FINE ? (lane & 48) | row : lane;           // the token of row lc of G^T; where a lane's token stands, four of a quarter side by side
  const int pt_n = a.P >> 4, unit = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  const int seg = unit / pt_n, pt = unit - seg * pt_n;
  if (seg >= (OUT ? a.nseg : a.nseg - 1)) return;                     // (no barrier in this kernel)
  const int c0 = seg * a.seg_chunks, c1 = min(c0 + a.seg_chunks, a.nch);
  const int g = a.group_map ? h % a.G : h / (a.H / a.G);
  const float* const xb = a.x + (int64_t)b * a.xsb + (int64_t)h * a.P + 16 * pt;
  const float* const Bb = a.Bm + (int64_t)b * a.bsb + (int64_t)g * a.bsg;
  const float* const Cb = a.Cm + (int64_t)b * a.csb + (int64_t)g * a.csg;
  const float* const db = a.dt + (int64_t)b * a.dsb + h;
  const float Ah = a.A[h], bias = a.dt_bias ? a.dt_bias[h] : 0.f, Dh = OUT && a.D ? a.D[h] : 0.f;
  const int64_t bh = (int64_t)b * a.H + h, nbh = (int64_t)gridDim.z * a.H, PN = (int64_t)a.P * FN;
  const int64_t mine = bh * PN + (16 * pt + lc) * FN + 4 * q;         // this lane's four state entries: column 16 pt + lc, n = 4 q ..

  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  float before = 0.f;
  if constexpr (OUT) {
    if (a.init) S = *(const f32x4*)(a.init + mine);
    if (seg > 0) {
      const float sd = lane < seg ? a.segdec[lane * nbh + bh] : 0.f, e = __expf(sd);
      for (int j0 = 0; j0 < seg; j0 += 8) {
        f32x4 v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = *(const f32x4*)(a.loc + min(j0 + j, seg - 1) * (nbh * PN) + mine);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j0 + j < seg) {
            const float f = rdlane(e, j0 + j);
#pragma unroll
            for (int r = 0; r < 4; ++r) S[r] = fmaf(f, S[r], v[j][r]);
          }
      }
      if (seg == a.nseg - 1) for (int j = 0; j < seg; ++j) before += rdlane(sd, j);
    }
  }
  float own = 0.f;
  for (int c = c0; c < c1; ++c) {
    const int t0 = c * FQ, tt = min(FQ, a.L - t0);
    const bool next = !OUT || c + 1 < c1 || (c + 1 == a.nch && a.final_state);        // the state behind this chunk is wanted
    const float raw = db[(int64_t)(t0 + min(lane, tt - 1)) * a.dsl];
    float xa[4][4], bn[4][4];
    f32x4 ba[4], ca[4], xd[4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t t = t0 + min(16 * st + tok(r), tt - 1);
        xa[st][r] = xb[t * a.xsl + lc];
        bn[st][r] = Bb[t * a.bsl + lc];
      }
    if constexpr (OUT) {
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int64_t t = t0 + min(16 * st + lc, tt - 1);
        ba[st] = *(const f32x4*)(Bb + (t0 + min(16 * st + row, tt - 1)) * a.bsl + 4 * q);
        ca[st] = *(const f32x4*)(Cb + t * a.csl + 4 * q);
        xd[st] = *(const f32x4*)(xb + t * a.xsl + 4 * q);
      }
    }
    float d = raw + bias;
    if (a.softplus) d = softplus_f(d);
    d = lane < tt ? fminf(fmaxf(d, a.dt_min), a.dt_max) : 0.f;
    const float da = d * Ah;
    if constexpr (FINE) {
      if (__ballot(!(da > -80.f && da < 1.f && d < 0x1p20f)) != 0) {
        own += march<OUT>(a, xb, Bb, Cb, t0, tt, d, da, Dh, lc, q, b, h, pt, S);
        continue;
      }
    }
    float lost = 0.f;
    const float cs = FINE ? scan_both(da, lost) : wave_incl_scan_dpp(da), cend = rdlane(cs, 63);      // (tokens past the end add 0)
    // what decays behind a token, summed from the end: cend - cs would carry the rounding of the whole chunk's sum into the tokens that weigh most
    float behind, behind_lost = 0.f;
    if constexpr (FINE) behind = scan_both(from_lane(da, 63 - lane), behind_lost);
    else behind = wave_incl_scan_dpp(from_lane(da, 63 - lane));
    const float back = from_lane(behind + behind_lost, 62 - lane);
    own += cend;
    sv[wave][0][slot] = cs;
    sv[wave][1][slot] = d;
    if constexpr (FINE) sv[wave][3][slot] = lost;
    sv[wave][2][slot] = lane == 63 ? d : exp_of<FINE>(back) * d;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                // (a wave's own LDS: in order)
    if (tt < FQ) {                                                    // rows past the end are zeros, as tokens that are not there
#pragma unroll
      for (int st = 0; st < 4; ++st) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * st + tok(r) >= tt) xa[st][r] = bn[st][r] = 0.f;
        if (OUT && 16 * st + row >= tt) ba[st] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    if constexpr (OUT) {
      float zero[4] = {};                                             // NaN where one of this wave's columns holds anything but numbers (0.5 % of the time)
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) zero[r] = fmaf(xa[st][r], 0.f, zero[r]);
      const bool odd = __ballot(zero[0] + zero[1] + (zero[2] + zero[3]) != 0.f) != 0;
      f32x4 css[4], ds[4], cls[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        css[st] = *(const f32x4*)&sv[wave][0][16 * st + 4 * q];
        if constexpr (FINE) cls[st] = *(const f32x4*)&sv[wave][3][16 * st + 4 * q];
        if constexpr (!FINE) ds[st] = *(const f32x4*)&sv[wave][1][16 * st + 4 * q];
        else ba[st] *= sv[wave][1][16 * st + lc];
      }
#pragma unroll
      for (int ot = 0; ot < 4; ++ot) {                                // 16 output tokens
        const float cst = sv[wave][0][16 * ot + row], clt = FINE ? sv[wave][FINE ? 3 : 0][16 * ot + row] : 0.f, et = __expf(cst);
        f32x4 Y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k) Y = mfma4(S[k], ca[ot][k], Y);
#pragma unroll
        for (int r = 0; r < 4; ++r) Y[r] *= et;
#pragma unroll
        for (int st = 0; st <= ot; ++st) {
          f32x4 M = {0.f, 0.f, 0.f, 0.f};
          if constexpr (FINE) {
            const f32x4 z = M;
            M = (mfma4(ba[st][0], ca[ot][0], z) + mfma4(ba[st][1], ca[ot][1], z)) + (mfma4(ba[st][2], ca[ot][2], z) + mfma4(ba[st][3], ca[ot][3], z));
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) M = mfma4(ba[st][k], ca[ot][k], M);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float gap = cst - css[st][r];
            if constexpr (FINE) gap += clt - cls[st][r];
            const float m = FINE ? __expf(gap) * M[r] : __expf(gap) * ds[st][r] * M[r];
            M[r] = st < ot || tok(r) <= lc ? m : 0.f;
          }
          if (st == ot && odd) {
            // (a factor of 0 does not hide an infinity or a NaN from the tokens in front of it: term by term)
#pragma unroll
            for (int t = 0; t < 16; ++t) {
              const float m = FINE ? from_lane(M[t >> 2], 16 * (t & 3) + lc) : from_lane(M[t & 3], 16 * (t >> 2) + lc);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float xt = from_lane(xd[ot][r], 16 * q + t);
                if (t <= lc) Y[r] = fmaf(xt, m, Y[r]);
              }
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) Y = mfma4(xa[st][r], M[r], Y);
          }
        }
        if (16 * ot + lc < tt) {
          f32x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = fmaf(Dh, xd[ot][r], Y[r]);
          *(f32x4*)(a.y + (int64_t)b * a.ysb + (int64_t)(t0 + 16 * ot + lc) * a.ysl + (int64_t)h * a.P + 16 * pt + 4 * q) = o;
        }
      }
    }
    if (next) {
      const float ec = exp_of<FINE>(cend);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] *= ec;
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const f32x4 w = *(const f32x4*)&sv[wave][2][16 * st + 4 * q];
#pragma unroll
        for (int r = 0; r < 4; ++r) S = mfma4(w[r] * bn[st][r], xa[st][r], S);
      }
    }
    asm volatile("" ::: "memory");                                    // (the next chunk's vectors are written behind this one's reads)
  }
  if constexpr (!OUT) {
    *(f32x4*)(a.loc + seg * (nbh * PN) + mine) = S;
    if (pt == 0 && lane == 0) a.segdec[seg * nbh + bh] = own;
  } else if (seg == a.nseg - 1) {
    if (a.final_state) *(f32x4*)(a.final_state + mine) = S;
    if (a.total_decay && pt == 0 && lane == 0) a.total_decay[bh] = before + own;
  }
}

// Chunks a segment: at most 64 segments (the fold keeps a segment's decay a lane), and the least of rounds of two waves a SIMD times a segment's chunks and .9 for what stands
// around them; a begun round counts .3 and its share of the rest.  (Rounded down to a round or more, us, before -> here, 32 heads x 64: 2 x 3 000 tokens 86 -> 66, 1 x 3 500:
// 57 -> 47, 2 x 1 300: 41 -> 38; 128 heads: 2 x 700: 80 -> 60, 2 x 2 100: 218 -> 159; always up: 1 x 2 100 36.0 | 38.2, 1 x 1 300: 27.1 | 28.1.  One wave a SIMD: 2 x 4 096: 92 | 105,
// four: 93.)
int chunks_a_segment(int batch, int nch, int nheads, int headdim) {
  const int64_t waves = (int64_t)batch * nheads * (headdim / 16), round = 8ll * tv_cu_count();
  const int64_t from = (nch + 63) / 64, most = waves * nch / round + 1, to = most < from ? from : most > nch ? nch : most;      // (from `most` on one round or less)
  int64_t best = from;
  double least = 1e300;
  for (int64_t len = from; len <= to; ++len) {
    const int64_t all = waves * ((nch + len - 1) / len), full = all / round;
    const double part = (double)(all % round) / round, rounds = full == 0 ? 1 : part > 0 ? full + .3 + .7 * part : full, t = rounds * (len + .9);
    if (t < least) { least = t; best = len; }
  }
  return (int)best;
}

}  // namespace

size_t tv_ssd_f32_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int dstate) {
  if (dstate != FN || headdim % 16 || batch <= 0 || seqlen <= 0 || nheads <= 0) return 0;
  const int nch = (seqlen + FQ - 1) / FQ, len = chunks_a_segment(batch, nch, nheads, headdim), nseg = (nch + len - 1) / len;
  return nseg == 1 ? 0 : (size_t)nseg * batch * nheads * ((size_t)headdim * FN + 1) * sizeof(float);
}

// called from ssd_chunked.hip and, beyond its lengths, from ssd_scan.hip: fp32 shapes whose rows are read and written in 16-byte pieces
bool tv_ssd_f32_supported(int headdim, int dstate, int64_t xsb, int64_t xsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg,
                          int64_t ysb, int64_t ysl, const void* x, const void* Bm, const void* Cm, const void* y, const void* init,
                          const void* final_state) {
  const int64_t strides = xsb | xsl | bsb | bsl | bsg | csb | csl | csg | ysb | ysl;
  const uintptr_t at = (uintptr_t)x | (uintptr_t)Bm | (uintptr_t)Cm | (uintptr_t)y | (uintptr_t)init | (uintptr_t)final_state;
  return dstate == FN && headdim % 16 == 0 && strides % 4 == 0 && at % 16 == 0;
}

int tv_ssd_f32_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* D, const void* dt_bias,
                      const void* init_state, void* y, void* final_state, void* total_decay, int batch, int seqlen, int nheads, int headdim, int ngroups,
                      int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg,
                      int64_t ysb, int64_t ysl, int dt_softplus, float dt_min, float dt_max, int group_map, bool fine, void* workspace, hipStream_t st) {
  F3Args a;
  a.x = (const float*)x; a.dt = (const float*)dt; a.Bm = (const float*)Bm; a.Cm = (const float*)Cm; a.A = (const float*)A; a.D = (const float*)D;
  a.dt_bias = (const float*)dt_bias; a.init = (const float*)init_state; a.y = (float*)y; a.final_state = (float*)final_state;
  a.total_decay = (float*)total_decay;
  a.L = seqlen; a.H = nheads; a.P = headdim; a.G = ngroups; a.nch = (seqlen + FQ - 1) / FQ;
  a.seg_chunks = chunks_a_segment(batch, a.nch, nheads, headdim);
  a.nseg = (a.nch + a.seg_chunks - 1) / a.seg_chunks;
  a.loc = (float*)workspace;
  a.segdec = a.loc + (int64_t)a.nseg * batch * nheads * headdim * FN;
  a.xsb = xsb; a.xsl = xsl; a.dsb = dsb; a.dsl = dsl; a.bsb = bsb; a.bsl = bsl; a.bsg = bsg; a.csb = csb; a.csl = csl; a.csg = csg; a.ysb = ysb; a.ysl = ysl;
  a.softplus = dt_softplus; a.group_map = group_map; a.dt_min = dt_min; a.dt_max = dt_max;
  const int units = headdim / 16 * a.nseg;
  const dim3 first((unsigned)((units - headdim / 16 + 3) / 4), (unsigned)nheads, (unsigned)batch);
  if (a.nseg > 1) {
    if (fine) ssd_f32_kernel<false, true><<<first, 256, 0, st>>>(a);
    else ssd_f32_kernel<false, false><<<first, 256, 0, st>>>(a);
  }
  const dim3 grid((unsigned)((units + 3) / 4), (unsigned)nheads, (unsigned)batch);
  if (fine) ssd_f32_kernel<true, true><<<grid, 256, 0, st>>>(a);
  else ssd_f32_kernel<true, false><<<grid, 256, 0, st>>>(a);
  TV_LAUNCH_CHECK();
}
