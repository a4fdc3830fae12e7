// S3 (fp32, d_state 16, head_dim a multiple of 16): the scan in blocks of 16 tokens on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 products
// and sums, 4 columns of contraction a step), one launch.
//
// A WAVE takes 16 columns of a head through a segment of the sequence, block by block, and nothing but the tokens' decays passes LDS, because the operands chain:
//   * G^T = B C^T puts, in a lane, four source tokens of one output token (rows 4 (lane / 16) + r, column lane % 16); numbering the four steps of a
//     contraction of 16 tokens the same way (step r, quarter q: token 4 q + r), M^T = decays x dt x G^T is the operand of Y^T += x^T M^T as it leaves G;
//   * the state S^T += (w B)^T x leaves, in a lane, four entries n of one column p: the operand of Y^T = S C^T as it is, and 16-byte rows in memory;
//   * Y^T leaves four neighbouring columns of one token: 16-byte stores.
// The waves of a work-group are the segments of one column tile: each forms the state that its segment leaves from a zero start, they meet once, each folds its
// predecessors' (in order, as the recurrence) and marches again, writing y.  Where the tiles leave half of the compute units idle, two work-groups share one: the second
// forms the first one's states again (a quarter of a chunk's work) instead of waiting for them.
// What bounds it is issue: vector, scalar and matrix instructions together take 1.1 of the SIMDs' cycles (4 096 tokens).  Hence blocks of 16 tokens: 64 products a chunk of 64 tokens
// (chunks of 64 as one tile take 112: G and its use grow with the square), a quarter of the exponentials, sums within 16 lanes; one rolled loop over all three passes, since a short call
// waits for its code (unrolled, with the next chunk's loads in flight: 64 tokens 7.0 us, 4 096: 50); addresses that move by scalar additions (64-bit products a load: 48 us for 43).
// Keeping all of a chunk's vectors in LDS for the last pass, not the steps alone, gives nothing (15.6 | 16.2 us at 1 024).
// Measured (32 heads x 64, 2 groups; two launches with chunks of 64 tokens -> here): 64 tokens 8.7 -> 6.7 us, 256: 12.6 -> 9.0, 1 024: 21.1 -> 15.6, 2 x 1 024: 30.0 -> 21.1,
// 4 096: 50 -> 43, 2 x 4 096: 87 -> 65, 8 192: 100 -> 82; 128 heads, 2 x 2 100: 159 -> 135.  Few heads and long sequences, or x beyond the last-level cache, which it reads twice: ssd_f32_long.hip
// (two_launches).  Error against 64 bits (exponents are differences of sums of 16 tokens, not of 64), fresh Mamba-2 layer, 1 024 tokens: y 2.5e-7 -> 1.1e-7, final state 1.0e-7 both.
#include "ssd_f32.hpp"

namespace {
using namespace ssdk;

constexpr int SEGS = 16;              // waves of a work-group at most
constexpr int KEEP = 4;               // chunks whose steps stay in LDS between a wave's passes

// sums over a block of 16 lanes, from its first lane on or (BACK) from its last, the lane's own among them; `lost`: what their rounding lost (an infinite sum has lost nothing)
template <bool FINE, bool BACK>
__device__ __forceinline__ float block_sum(float v, float& lost) {
  constexpr int SH = BACK ? 0x100 : 0x110;      // row_shl, row_shr
  lost = 0.f;
  if constexpr (FINE) {
    scan_step<SH + 1, 0xf>(v, lost);
    scan_step<SH + 2, 0xf>(v, lost);
    scan_step<SH + 4, 0xf>(v, lost);
    scan_step<SH + 8, 0xf>(v, lost);
    lost = fabsf(v) < INFINITY ? lost : 0.f;
  } else {
    v += dpp_shift<SH + 1, 0xf>(v);
    v += dpp_shift<SH + 2, 0xf>(v);
    v += dpp_shift<SH + 4, 0xf>(v);
    v += dpp_shift<SH + 8, 0xf>(v);
  }
  return v;
}

// FINE: for the lengths that the token recurrence had before (48 - 64 tokens, more than 4 096), whose error and whose results at extreme steps are kept:
//   * two tokens' decay is the difference of their sums AND of what these have lost (a sum over a chunk is rounded by its own size, not by the difference's);
//   * the four steps of a contraction of 16 tokens are numbered in time (step r, quarter q: token 4 r + q; the rows of G^T are dealt out to match), so that what weighs most is added
//     last and rounded once, as by the recurrence; B has dt, and its sum with C over n is a tree;
//   * the decays of the state's weights are sums that keep what they lose, and their exponentials are the recurrence's own;
//   * a chunk with a token that leaves nothing of what was before it (dt A below -80, an infinite dt among them), or whose dt or dt A is otherwise out of the ordinary, goes token by
//     token (dt B, sums of dt A and differences of them are infinite or NaN there while the recurrence's products are not).
// Error against 64 bits, recurrence | here, 64 tokens of 32 heads x 64 that decay by e^-52: y 7.5e-8 | 7.2e-8, state 6.0e-8 | 5.7e-8; by e^-15: 8.8e-8 | 8.6e-8, 7.0e-8 | 6.7e-8; slowly:
// 2.2e-7 | 1.4e-7, 2.8e-7 | 1.6e-7; 5 000 tokens: 7.3e-8 | 6.9e-8, 6.1e-8 | 5.5e-8, slowly 4.0e-6 | 3.7e-7 (steps numbered as at the other lengths: 8.4e-8 for the first).
template <bool FINE>
__global__ __launch_bounds__(64 * SEGS) void ssd_f32_kernel(F3Args a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char f3_smem[];
  const int nw = (int)(blockDim.x >> 6);
  typedef float Vec[FQ];
  Vec(*const sv)[4] = (Vec(*)[4])f3_smem;                                        // a wave's own: cs, dt, weights of the state, what cs has lost
  Vec(*const kd)[KEEP] = (Vec(*)[KEEP])(sv + nw);                                // a wave's own: dt behind the softplus, of its first chunks
  f32x4(*const left)[64] = (f32x4(*)[64])(kd + nw);                              // the states that segments leave from a zero start, in their order
  float* const segd = (float*)(left + 2 * nw);                                   // and their sums of dt A
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 15, q = lane >> 4;
  auto tok = [&](int r) __attribute__((always_inline)) { return FINE ? 4 * r + q : 4 * q + r; };       // of the 16: step r's token in this quarter
  const int row = FINE ? (lc & 3) << 2 | lc >> 2 : lc, slot = FINE ? (lane & 48) | row : lane;           // the token of row lc of G^T; where a lane's token stands, four of a quarter side by side
  const int h = blockIdx.x, pt = blockIdx.y;                                     // (column tiles of a head on one XCD, where eight divides the heads: they share lines of x, and B and C)
  // chunks [from, to) are this work-group's, `len` a segment and wave; those in front of them give it a state only, `plen` a segment, from its last wave on
  const int b = a.two ? blockIdx.z >> 1 : blockIdx.z;
  const bool second = a.two && (blockIdx.z & 1);
  const int from = second ? a.split : 0, to = second || !a.two ? a.nch : a.split, len = second ? a.len1 : a.len0, npre = second ? a.npre : 0;
  const int c0 = from + wave * len, c1 = min(c0 + len, to);                      // (c0 >= c1: none)
  const bool last = c1 == a.nch && c0 < c1;
  const int g = a.group_map ? h % a.G : h / a.hpg;
  const float* const xb = a.x + (int64_t)b * a.xsb + (int64_t)h * a.P + 16 * pt;
  const float* const Bb = a.Bm + (int64_t)b * a.bsb + (int64_t)g * a.bsg;
  const float* const Cb = a.Cm + (int64_t)b * a.csb + (int64_t)g * a.csg;
  const float* const db = a.dt + (int64_t)b * a.dsb + h;
  const float Ah = a.A[h], bias = a.dt_bias ? a.dt_bias[h] : 0.f, Dh = a.D ? a.D[h] : 0.f;
  const int64_t bh = (int64_t)b * a.H + h, mine = bh * a.P * FN + (16 * pt + lc) * FN + 4 * q;         // this lane's four state entries: column 16 pt + lc, n = 4 q ..

  // rows of a chunk at 32-bit offsets from its first
  typedef __attribute__((address_space(1))) const unsigned char* gp;
  auto at1 = [](const float* base, unsigned off) __attribute__((always_inline)) { return *(__attribute__((address_space(1))) const float*)((gp)base + off); };
  auto at4 = [](const float* base, unsigned off) __attribute__((always_inline)) { return *(__attribute__((address_space(1))) const f32x4*)((gp)base + off); };
  auto down = [](const float* p, int bytes) __attribute__((always_inline)) { return (const float*)((const unsigned char*)p + (unsigned)bytes); };
  const int xs4 = (int)a.xsl * 4, bs4 = (int)a.bsl * 4, cs4 = (int)a.csl * 4, ys4 = (int)a.ysl * 4;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  // ---- a block of 16 tokens: x and B, a token a step of the contraction; rows of B, C and x.  Those of the block behind are asked for ahead
  struct Block {
    float xa[4], bn[4];
    f32x4 ba, ca, xd;
  };
  unsigned ox[4], ob[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    ox[r] = (unsigned)(tok(r) * xs4 + 4 * lc);
    ob[r] = (unsigned)(tok(r) * bs4 + 4 * lc);
  }
  const float *xc, *bc, *cc;                                          // first rows of the block that is asked for next
  int ahead;                                                          // tokens from there on
  auto start = [&](int c) __attribute__((always_inline)) {
    xc = xb + (int64_t)(c * FQ) * a.xsl;
    bc = Bb + (int64_t)(c * FQ) * a.bsl;
    cc = Cb + (int64_t)(c * FQ) * a.csl;
    ahead = a.L - c * FQ;
  };
  auto load = [&](bool out) __attribute__((always_inline)) {
    Block B;
    const int end = min(15, ahead - 1);
    if (end == 15) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        B.xa[r] = at1(xc, ox[r]);
        B.bn[r] = at1(bc, ob[r]);
      }
    } else {                                                          // rows past the end are zeros, as tokens that are not there
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = tok(r), u = min(t, end);
        const float v = at1(xc, (unsigned)(u * xs4 + 4 * lc)), w = at1(bc, (unsigned)(u * bs4 + 4 * lc));
        B.xa[r] = t <= end ? v : 0.f;
        B.bn[r] = t <= end ? w : 0.f;
      }
    }
    if (out) {
      B.ba = at4(bc, (unsigned)(min(row, end) * bs4 + 16 * q));
      B.ca = at4(cc, (unsigned)(min(lc, end) * cs4 + 16 * q));
      B.xd = at4(xc, (unsigned)(min(lc, end) * xs4 + 16 * q));
      if (row > end) B.ba = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    xc = down(xc, 16 * xs4);
    bc = down(bc, 16 * bs4);
    cc = down(cc, 16 * cs4);
    ahead -= 16;
    return B;
  };
  // ---- a chunk's tokens, one a lane
  float d, da, cend, ecs;                                             // ecs: what is left behind a block's last token (lanes 15, 31, ..) of what was in front of the block
  bool odd_steps = false;
  auto load_dt = [&](int c) __attribute__((always_inline)) { return db[(int64_t)min(c * FQ + lane, a.L - 1) * a.dsl]; };
  // kept: d is what raw says, of the pass in front
  auto prep = [&](int c, float raw, bool kept) __attribute__((always_inline)) {
    d = raw;
    if (!kept) {
      d += bias;
      if (a.softplus) d = softplus_f(d);
      d = lane < a.L - c * FQ ? fminf(fmaxf(d, a.dt_min), a.dt_max) : 0.f;
    }
    da = d * Ah;
    if constexpr (FINE) {
      odd_steps = __ballot(!(da > -80.f && da < 1.f && d < 0x1p20f)) != 0;
      if (odd_steps) return;
    }
    float lost, back_lost;
    const float cs = block_sum<FINE, false>(da, lost);                // (tokens past the end add 0)
    cend = (rdlane(cs, 15) + rdlane(cs, 31)) + (rdlane(cs, 47) + rdlane(cs, 63));
    // what decays behind a token, summed from the end: a difference of sums would carry the rounding of the whole block's into the tokens that weigh most
    const float behind = block_sum<FINE, true>(da, back_lost);
    const float back = dpp_shift<0x101, 0xf>(behind + back_lost);
    ecs = exp_of<FINE>(cs);
    sv[wave][0][slot] = cs;
    sv[wave][1][slot] = d;
    if constexpr (FINE) sv[wave][3][slot] = lost;
    sv[wave][2][slot] = (lane & 15) == 15 ? d : exp_of<FINE>(back) * d;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                // (a wave's own LDS: in order)
  };
  auto pass_state = [&](const Block& B, int k) __attribute__((always_inline)) {       // the state behind block k of a chunk
    const float ec = rdlane(ecs, 16 * k + 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] *= ec;
    const f32x4 w = *(const f32x4*)&sv[wave][2][16 * k + 4 * q];
#pragma unroll
    for (int r = 0; r < 4; ++r) S = mfma4(w[r] * B.bn[r], B.xa[r], S);
  };
  // the outputs of block k of a chunk from the state in front of it
  float* yc = nullptr;                                                // first row of the block
  const unsigned oy = (unsigned)(lc * ys4 + 16 * q);
  auto outputs = [&](const Block& B, int k, int tt) __attribute__((always_inline)) {
    float zero = 0.f;                                                 // NaN where one of this wave's columns holds anything but numbers
#pragma unroll
    for (int r = 0; r < 4; ++r) zero = fmaf(B.xa[r], 0.f, zero);
    const bool odd = __ballot(zero != 0.f) != 0;
    const float cst = sv[wave][0][16 * k + row], clt = FINE ? sv[wave][FINE ? 3 : 0][16 * k + row] : 0.f, et = __expf(cst);
    const f32x4 css = *(const f32x4*)&sv[wave][0][16 * k + 4 * q];
    f32x4 Y = {0.f, 0.f, 0.f, 0.f}, M = Y, ds, cls, bk = B.ba;
    if constexpr (FINE) {
      cls = *(const f32x4*)&sv[wave][3][16 * k + 4 * q];
      bk *= sv[wave][1][16 * k + lc];
      const f32x4 z = Y;
      M = (mfma4(bk[0], B.ca[0], z) + mfma4(bk[1], B.ca[1], z)) + (mfma4(bk[2], B.ca[2], z) + mfma4(bk[3], B.ca[3], z));
    } else {
      ds = *(const f32x4*)&sv[wave][1][16 * k + 4 * q];
#pragma unroll
      for (int n = 0; n < 4; ++n) M = mfma4(bk[n], B.ca[n], M);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) Y = mfma4(S[n], B.ca[n], Y);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Y[r] *= et;
      float gap = cst - css[r];
      if constexpr (FINE) gap += clt - cls[r];
      const float m = FINE ? __expf(gap) * M[r] : __expf(gap) * ds[r] * M[r];
      M[r] = tok(r) <= lc ? m : 0.f;
    }
    if (odd) {
      // (a factor of 0 does not hide an infinity or a NaN from the tokens in front of it: term by term)
#pragma unroll 1
      for (int t = 0; t < 16; ++t) {
        const int i = FINE ? t >> 2 : t & 3;
        const float m = from_lane(i < 2 ? (i ? M[1] : M[0]) : (i == 2 ? M[2] : M[3]), 16 * (FINE ? t & 3 : t >> 2) + lc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float xt = from_lane(B.xd[r], 16 * q + t);
          if (t <= lc) Y[r] = fmaf(xt, m, Y[r]);
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) Y = mfma4(B.xa[r], M[r], Y);
    }
    if (lc < tt) {
      f32x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = fmaf(Dh, B.xd[r], Y[r]);
      *(__attribute__((address_space(1))) f32x4*)((__attribute__((address_space(1))) unsigned char*)yc + oy) = o;
    }
    yc = (float*)down(yc, 16 * ys4);
  };

  // ---- three passes of one loop (its code is what a short call waits for): what a segment in front of this work-group's chunks leaves from a zero start, what this wave's
  // own leaves, and then, from the state that enters it, its outputs
  const int pre = nw - 1 - wave;
  float before = 0.f, own = 0.f;
#pragma unroll 1
  for (int pass = 0; pass < 3; ++pass) {
    const bool out = pass == 2;
    int lo = c0, hi = c1, to_left = npre + wave;
    if (pass == 0) {
      lo = pre * a.plen;
      hi = pre < npre ? min(lo + a.plen, from) : lo;
      to_left = pre;
    } else if (pass == 1 && c1 == to) {                               // (nobody behind it)
      hi = lo;
    }
    if (out) __syncthreads();
    if (lo >= hi) continue;
    start(lo);
    // (the steps of this wave's first chunks stay where they are from one pass to the next)
    const int keep = pass != 0 && c1 < to ? KEEP : 0;
    float raw = out && keep ? 0.f : load_dt(lo);
    Block B = load(out);
    if (out) yc = a.y + (int64_t)b * a.ysb + (int64_t)(lo * FQ) * a.ysl + (int64_t)h * a.P + 16 * pt;
    S = f32x4{0.f, 0.f, 0.f, 0.f};
    own = 0.f;
    if (out) {                                                        // the initial state and the segments in front, folded in their order
      if (a.init) S = *(const f32x4*)(a.init + mine);
      const int front = npre + wave;
      if (front > 0) {
        const float sd = lane < front ? segd[lane] : 0.f, e = __expf(sd);
        for (int j0 = 0; j0 < front; j0 += 4) {
          f32x4 v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = left[min(j0 + j, front - 1)][lane];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (j0 + j < front) {
              const float f = rdlane(e, j0 + j);
#pragma unroll
              for (int r = 0; r < 4; ++r) S[r] = fmaf(f, S[r], v[j][r]);
            }
        }
        if (last) for (int j = 0; j < front; ++j) before += rdlane(sd, j);
      }
    }
#pragma unroll 1
    for (int c = lo; c < hi; ++c) {
      const bool kept = out && c - lo < keep;
      prep(c, kept ? kd[wave][(c - lo) & (KEEP - 1)][lane] : raw, kept);
      if (!out && c - lo < keep) kd[wave][(c - lo) & (KEEP - 1)][lane] = d;
      if (c + 1 < hi && !(out && c + 1 - lo < keep)) raw = load_dt(c + 1);
      if (FINE && odd_steps) {
        const int tt = min(FQ, a.L - c * FQ);
        own += out ? march<true>(a, xb, Bb, Cb, c * FQ, tt, d, da, Dh, lc, q, b, h, pt, S) : march<false>(a, xb, Bb, Cb, c * FQ, tt, d, da, Dh, lc, q, b, h, pt, S);
        if (c + 1 < hi) {
          start(c + 1);
          B = load(out);
          if (out) yc = a.y + (int64_t)b * a.ysb + (int64_t)((c + 1) * FQ) * a.ysl + (int64_t)h * a.P + 16 * pt;
        }
        continue;
      }
      own += cend;
      const int tt = min(FQ, a.L - c * FQ), blocks = (tt + 15) >> 4;
#pragma unroll 1
      for (int k = 0; k < blocks; ++k) {
        const Block N = k + 1 < blocks || c + 1 < hi ? load(out) : B;
        if (out) outputs(B, k, tt - 16 * k);
        pass_state(B, k);
        B = N;
      }
    }
    if (!out) {
      left[to_left][lane] = S;
      if (lane == 0) segd[to_left] = own;
    }
  }
  if (c0 >= c1) return;
  if (last) {
    if (a.final_state) *(f32x4*)(a.final_state + mine) = S;
    if (a.total_decay && pt == 0 && lane == 0) a.total_decay[bh] = before + own;
  }
}

// Waves a work-group, chunks of the first of two work-groups (all: there is one), chunks a segment of the first and the second one's own and of those that the second forms again
struct F3Plan {
  int waves, split, len0, len1, plen;
};
// Four waves a SIMD, of 16 a work-group at most (16 | 8 waves, us: 1 024 tokens 15.6 | 16.9, 4 096: 43 | 49).  Two work-groups a tile where one would leave half of the compute
// units idle (1 024 tokens 18.3 | 15.6, 4 096: 71 | 43; 2 x 1 024, where it would not: 21.1 | 26), from 8 chunks on; the first has 9/16 of the chunks: a state takes a quarter to a third of what
// outputs and state together do.
F3Plan plan(int batch, int nch, int nheads, int headdim) {
  const int64_t units = (int64_t)batch * nheads * (headdim / 16), full = (16ll * tv_cu_count() + units - 1) / units;
  const bool two = 2 * units <= tv_cu_count() && nch >= 8;
  auto up = [](int n, int d) { return (n + d - 1) / d; };
  F3Plan p;
  p.waves = (int)(full < SEGS ? full : SEGS);
  if (p.waves > nch) p.waves = nch;
  p.split = two ? up(9 * nch, 16) : nch;
  p.len0 = up(p.split, p.waves);
  p.len1 = two ? up(nch - p.split, p.waves) : 1;
  p.plen = p.len0;
  return p;
}

// Whether two launches on longer segments (ssd_f32_long.hip) are the faster ones.  Timed (us, here | there) over 36 shapes of 8 to 6 144 column tiles (batch x heads x head_dim / 16) and
// 128 to 40 000 tokens:
//   * few tiles: 32 segments a tile at most leave the chip idle.  Up to 32 tiles from 24 chunks on (16 tiles, 1 024 tokens 13.9 | 14.8, 1 500: 18.4 | 17.7), up to 64 from 60 on (64:
//     3 000 tokens 32.4 | 38.0, 4 096: 41.6 | 40.3), up to 80 beyond 64 chunks (80, 8 192: 84 | 79).
//   * up to 4 096 tokens, where FINE costs there what it does not here, else only 1 792 to 2 559 tiles with more than 240 MB of x (2 048: 326 | 312, 4 096 tokens 677 | 617).
//   * longer ones where x, read again by the second half of a tile's work-groups and by every segment, is not in the last-level cache any more; how many MB that takes depends on how the
//     tiles fill their rounds.  128 tiles: 134 MB 161 | 195, 197 MB 316 | 299, 328 MB 583 | 501; 192: 101 MB 132 | 154, 201 MB 347 | 314; 256: 197 MB 267 | 291, 268 MB 420 | 406; 384: 147 MB
//     208 | 209, 403 MB 765 | 594; 640: 492 MB 773 | 750; 1 024: 197 MB 230 - 259 | 247, 537 MB 710 - 824 | 700; 2 048: 537 MB 677 - 692 | 580; 3 072 and more, which read x once, never.
//   * 129 to 159 tiles, half of a round that a second work-group a tile does not fit, from 120 chunks on (132: 6 000 tokens 84 | 87, 8 192: 113 | 108), 257 to 336, just over a round, from
//     65 on (264: 6 000: 169 | 160).
bool two_launches(int batch, int nch, int nheads, int headdim) {
  const int64_t tiles = (int64_t)batch * nheads * (headdim / 16);
  const double mb = 1e-6 * tiles * 16 * sizeof(float) * FQ * nch;
  if (tiles <= 32) return nch >= 24;
  if (tiles <= 64) return nch >= 60;
  if (nch <= 64) return tiles >= 1792 && tiles < 2560 && mb > 240;
  if (tiles <= 80) return true;
  if (tiles > 128 && tiles < 160) return nch >= 120;
  if (tiles > 256 && tiles <= 336) return true;
  static constexpr int LINE[][2] = {{128, 140}, {255, 120}, {256, 240}, {415, 190}, {831, 400}, {1151, 210}, {1791, 380}, {2559, 150}};     // tiles up to, MB
  for (const auto& l : LINE)
    if (tiles <= l[0]) return mb > l[1];
  return false;
}

}  // namespace

size_t tv_ssd_f32_long_workspace_bytes(int batch, int nch, int nheads, int headdim);
int tv_ssd_f32_long_launch(ssdk::F3Args a, int batch, void* workspace, hipStream_t st);

// What the launch can use; with less it is one launch
size_t tv_ssd_f32_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int dstate) {
  if (dstate != FN || headdim % 16 || batch <= 0 || seqlen <= 0 || nheads <= 0 || headdim <= 0) return 0;
  const int nch = (seqlen + FQ - 1) / FQ;
  return two_launches(batch, nch, nheads, headdim) ? tv_ssd_f32_long_workspace_bytes(batch, nch, nheads, headdim) : 0;
}

// called from ssd_chunked.hip and, beyond its lengths, from ssd_scan.hip: fp32 shapes whose rows are read and written in 16-byte pieces
bool tv_ssd_f32_supported(int headdim, int dstate, int64_t xsb, int64_t xsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg,
                          int64_t ysb, int64_t ysl, const void* x, const void* Bm, const void* Cm, const void* y, const void* init,
                          const void* final_state) {
  // (rows of a chunk at 32-bit offsets)
  for (const int64_t l : {xsl, bsl, csl, ysl})
    if (l < 0 || l * FQ * (int64_t)sizeof(float) >= (1ll << 31)) return false;
  const int64_t strides = xsb | xsl | bsb | bsl | bsg | csb | csl | csg | ysb | ysl;
  const uintptr_t at = (uintptr_t)x | (uintptr_t)Bm | (uintptr_t)Cm | (uintptr_t)y | (uintptr_t)init | (uintptr_t)final_state;
  return dstate == FN && headdim % 16 == 0 && strides % 4 == 0 && at % 16 == 0;
}

int tv_ssd_f32_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* D, const void* dt_bias,
                      const void* init_state, void* y, void* final_state, void* total_decay, int batch, int seqlen, int nheads, int headdim, int ngroups,
                      int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg,
                      int64_t ysb, int64_t ysl, int dt_softplus, float dt_min, float dt_max, int group_map, bool fine, void* workspace, size_t workspace_bytes, hipStream_t st) {
  F3Args a;
  a.x = (const float*)x; a.dt = (const float*)dt; a.Bm = (const float*)Bm; a.Cm = (const float*)Cm; a.A = (const float*)A; a.D = (const float*)D;
  a.dt_bias = (const float*)dt_bias; a.init = (const float*)init_state; a.y = (float*)y; a.final_state = (float*)final_state;
  a.total_decay = (float*)total_decay;
  a.L = seqlen; a.H = nheads; a.P = headdim; a.G = ngroups; a.nch = (seqlen + FQ - 1) / FQ;
  a.hpg = nheads / ngroups;
  a.xsb = xsb; a.xsl = xsl; a.dsb = dsb; a.dsl = dsl; a.bsb = bsb; a.bsl = bsl; a.bsg = bsg; a.csb = csb; a.csl = csl; a.csg = csg; a.ysb = ysb; a.ysl = ysl;
  a.softplus = dt_softplus; a.group_map = group_map; a.dt_min = dt_min; a.dt_max = dt_max;
  if (two_launches(batch, a.nch, nheads, headdim) && workspace_bytes >= tv_ssd_f32_long_workspace_bytes(batch, a.nch, nheads, headdim))
    return tv_ssd_f32_long_launch(a, batch, workspace, st);
  const F3Plan p = plan(batch, a.nch, nheads, headdim);
  a.two = p.split < a.nch; a.split = p.split; a.len0 = p.len0; a.len1 = p.len1; a.plen = p.plen;
  a.npre = (p.split + p.plen - 1) / p.plen;
  const dim3 grid((unsigned)nheads, (unsigned)(headdim / 16), (unsigned)(a.two ? 2 * batch : batch)), threads((unsigned)(64 * p.waves));
  const unsigned lds = (unsigned)p.waves * (unsigned)((4 + KEEP) * FQ * sizeof(float) + 2 * 64 * sizeof(f32x4) + 2 * sizeof(float));
  static const hipError_t attr = [] {
    const hipError_t e = hipFuncSetAttribute((const void*)ssd_f32_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
    return e != hipSuccess ? e : hipFuncSetAttribute((const void*)ssd_f32_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
  }();
  if (attr != hipSuccess) {
    tv_set_error("ssd_f32: cannot reserve %u bytes of LDS: %s", lds, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  if (fine) ssd_f32_kernel<true><<<grid, threads, lds, st>>>(a);
  else ssd_f32_kernel<false><<<grid, threads, lds, st>>>(a);
  TV_LAUNCH_CHECK();
}
