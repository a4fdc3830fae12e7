// The fp32 scan of ssd_f32.hip in two launches, for sequences that its one launch has too few waves for (few heads) or whose x does not stay in the last-level cache between that
// one's two readings; the line is two_launches() there.
//
// A wave takes 16 columns of a head through a segment of chunks of 64 tokens, with the same chain of operands, but a chunk as one tile: all its loads are asked for at once (what bounds
// these sequences is memory, or one wave's latencies), and the products with M grow to 40 of 112 a chunk.  First launch: the state that every segment but the last leaves from a zero
// start; second: a segment folds its predecessors' (in order, as the recurrence; 1 KB a predecessor and wave) and marches, writing y once.  How long a segment is: chunks_a_segment.
// The sums, their numbering and the chunks with extreme steps are as at FINE there: error against 64 bits of y 5e-8 to 9e-8 (fresh Mamba-2 decays), the one launch's 5e-8 to 1.6e-7.
// Measured (us, one launch | here): 8 heads x 32: 2 048 tokens 23.7 | 19.3, 4 096: 38.7 | 23.0, 16 384: 140 | 44, 60 000: 500 | 120; 16 x 64: 8 192: 79 | 63, 60 000: 732 | 390; 32 x 64:
// 16 384: 173 | 211 (left), 30 000: 435 | 394; 128 x 64 x 8 192, batch 4: 1 440 | 1 166; 128 x 128, 16 384: 1 430 | 1 380.
#include "ssd_f32.hpp"

namespace {
using namespace ssdk;

// inclusive sums over the lanes as value + what its rounding lost (an infinite sum has lost nothing)
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

// OUT: the second launch
template <bool OUT>
__global__ __launch_bounds__(256) void ssd_f32_long_kernel(F3Args a) {
  __shared__ __attribute__((aligned(16))) float sv[4][4][FQ];         // a wave's own: cs, dt, weights of the state, what cs has lost
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, q = lane >> 4;
  auto tok = [&](int r) __attribute__((always_inline)) { return 4 * r + q; };       // of the 16: step r's token in this quarter
  const int row = (lc & 3) << 2 | lc >> 2, slot = (lane & 48) | row;           // the token of row lc of G^T; where a lane's token stands, four of a quarter side by side
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
    if (__ballot(!(da > -80.f && da < 1.f && d < 0x1p20f)) != 0) {
      own += march<OUT>(a, xb, Bb, Cb, t0, tt, d, da, Dh, lc, q, b, h, pt, S);
      continue;
    }
    float lost, behind_lost;
    const float cs = scan_both(da, lost), cend = rdlane(cs, 63);      // (tokens past the end add 0)
    // what decays behind a token, summed from the end: cend - cs would carry the rounding of the whole chunk's sum into the tokens that weigh most
    const float behind = scan_both(from_lane(da, 63 - lane), behind_lost);
    const float back = from_lane(behind + behind_lost, 62 - lane);
    own += cend;
    sv[wave][0][slot] = cs;
    sv[wave][1][slot] = d;
    sv[wave][3][slot] = lost;
    sv[wave][2][slot] = lane == 63 ? d : expf(back) * d;
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
      f32x4 css[4], cls[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        css[st] = *(const f32x4*)&sv[wave][0][16 * st + 4 * q];
        cls[st] = *(const f32x4*)&sv[wave][3][16 * st + 4 * q];
        ba[st] *= sv[wave][1][16 * st + lc];
      }
#pragma unroll
      for (int ot = 0; ot < 4; ++ot) {                                // 16 output tokens
        const float cst = sv[wave][0][16 * ot + row], clt = sv[wave][3][16 * ot + row], et = __expf(cst);
        f32x4 Y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k) Y = mfma4(S[k], ca[ot][k], Y);
#pragma unroll
        for (int r = 0; r < 4; ++r) Y[r] *= et;
#pragma unroll
        for (int st = 0; st <= ot; ++st) {
          const f32x4 z = {0.f, 0.f, 0.f, 0.f};
          f32x4 M = (mfma4(ba[st][0], ca[ot][0], z) + mfma4(ba[st][1], ca[ot][1], z)) + (mfma4(ba[st][2], ca[ot][2], z) + mfma4(ba[st][3], ca[ot][3], z));
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float gap = (cst - css[st][r]) + (clt - cls[st][r]), m = __expf(gap) * M[r];
            M[r] = st < ot || tok(r) <= lc ? m : 0.f;
          }
          if (st == ot && odd) {
            // (a factor of 0 does not hide an infinity or a NaN from the tokens in front of it: term by term)
#pragma unroll
            for (int t = 0; t < 16; ++t) {
              const float m = from_lane(M[t >> 2], 16 * (t & 3) + lc);
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
      const float ec = expf(cend);
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
// 57 -> 47; 128 heads: 2 x 700: 80 -> 60, 2 x 2 100: 218 -> 159; always up: 1 x 2 100 36.0 | 38.2.  One wave a SIMD: 2 x 4 096: 92 | 105, four: 93.)
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

size_t tv_ssd_f32_long_workspace_bytes(int batch, int nch, int nheads, int headdim) {
  const int len = chunks_a_segment(batch, nch, nheads, headdim), nseg = (nch + len - 1) / len;
  return nseg == 1 ? 0 : (size_t)nseg * batch * nheads * ((size_t)headdim * FN + 1) * sizeof(float);
}

// called from ssd_f32.hip, with what both kernels read in `a`
int tv_ssd_f32_long_launch(ssdk::F3Args a, int batch, void* workspace, hipStream_t st) {
  a.seg_chunks = chunks_a_segment(batch, a.nch, a.H, a.P);
  a.nseg = (a.nch + a.seg_chunks - 1) / a.seg_chunks;
  a.loc = (float*)workspace;
  a.segdec = a.loc + (int64_t)a.nseg * batch * a.H * a.P * FN;
  const int units = a.P / 16 * a.nseg;
  if (a.nseg > 1) {
    ssd_f32_long_kernel<false><<<dim3((unsigned)((units - a.P / 16 + 3) / 4), (unsigned)a.H, (unsigned)batch), 256, 0, st>>>(a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      tv_set_error("ssd_f32: %s", hipGetErrorString(e));
      return TV_ERR_LAUNCH;
    }
  }
  ssd_f32_long_kernel<true><<<dim3((unsigned)((units + 3) / 4), (unsigned)a.H, (unsigned)batch), 256, 0, st>>>(a);
  TV_LAUNCH_CHECK();
}
