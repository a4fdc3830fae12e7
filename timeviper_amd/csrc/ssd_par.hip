// S3, middle lengths and batches: ONE HEAD PER WORK-GROUP, segments that start from the true state.
//
// A march over a few dozen chunks is a chain that hides nothing: 24 steps of 2.6 - 3.9 us on 160 work-groups were 85 us at 1 501 tokens, while its 70 MB
// take 14.  So the chain is cut into segments, and what enters a segment is formed first:
//   local    every segment but the last, from a zero state: the state it leaves (fp32, in the order of the registers that hold it) and its decay
//   output   every segment: the entering state is summed from the local states in front of it (until 2^-64 of one is left), then the march
// Two launches; y is written once.  Both are the same march over a head's chunks of 64 tokens:
//   * wave w of four holds rows n = 32 w .. + 31 of the state (40 registers at head_dim 80); its slice of B is its own, so B goes through a wave-private
//     tile (transposing reads) without a barrier;
//   * x is weighted once, x~_s = 2^(cs_e - cs_s) dt_s x_s (e: the chunk's last token; a factor <= 1), for all four waves and for both of its uses:
//     X := 2^cs_e X, y_t = 2^(cs_t - cs_e) (C_t . X + sum_{s <= t} CB[t][s] x~_s) + D x_t, X += B^T x~.  C . X takes all rows of X: as a bf16 copy in LDS, left at
//     the end of the step in front; wave w forms the 16 tokens 16 w .. of the chunk's outputs.  One barrier a step (two buffers);
//   * a chunk that decays by more than 2^100: everything 2^100 up for this chunk; by more than 2^199: x as it is in LDS, the true mask 2^(cs_t - cs_s) dt_s on
//     C.B^T, factors of x in registers for the state.  The row factor stays within 2^(+-100); no kind of chunk costs more than 10 % more than another.
// Rows of a pair of 16-row tiles are numbered 8 (r >> 2) + 4 half + (r & 3): a lane's eight results of a pair lie side by side (the state's copy is
// an operand as it leaves the registers).  Loads and stores take whole rows by neighbouring lanes and change layout in LDS: the results' own layout
// (16 rows a quarter wave) took 3 470 L1 accesses a step instead of 1 450.
// 80 KB of LDS and 252 registers: two work-groups a CU.  A step takes 3 us alone and 5 us beside another one: 380 vector, 48 matrix and 85 LDS
// instructions of a wave, which are busy a third of the time; the rest is their latencies (no phase stands out).
// Measured (128 heads x 80, 8 groups, whole operator without C.B^T): 512 tokens 31 -> 26 us, 1 501: 85 -> 50, 4 200: 143 -> 115; the rule's comment in ssd_head.hip
// has more sizes.
#include "ssd_common.hpp"

namespace {
using namespace ssdk;

constexpr int PQ = 64, PN = 128, PFR = 6;      // tokens a chunk, d_state, causal fragments of C.B^T a chunk
constexpr float LOG2E = 1.4426950408889634f;
constexpr float UP = 100.f, MASK_FROM = 199.f;  // log2 decays of a chunk: raised from here on, true mask from here on
constexpr float FORGOTTEN = -64.f;             // log2 of the factor from which on an earlier state is left out (as the march's resets)

struct ParArgs {
  const bf16_t *x, *dt, *Bm, *Cm, *cb;
  const float *A, *D, *dt_bias, *init;
  bf16_t* y;
  float *final_state, *total_decay;
  float *loc, *segdec;                         // [segment][batch][head]: local states in register order, sums of dt A
  int L, H, G, nchunks, nseg, seg_chunks;
  int64_t xsb, xsl, dsb, dsl, bsb, bsl, bsg, csb, csl, csg, ysb, ysl;
  int softplus, group_map;
  float dt_min, dt_max;
};

typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int XPAIR = PQ * 64 + 64;            // bytes of a pair of column tiles (32 columns) of a chunk of x
template <int PT, bool OUT>
struct __attribute__((aligned(16))) ParSmem {
  unsigned char x[2][(PT / 2) * XPAIR + (PT & 1) * PQ * 32];
  unsigned char b[4][PQ * 64];                 // a wave's own: its 16 rows of C, its 32 columns of B, its 16 rows of x and of y, one after the other
  bf16_t snap[OUT ? 2 : 1][OUT ? PT * 4 * 64 * 8 : 8];   // [column tile][quarter of the state rows][lane] 16 bytes
  float dt[2][PQ];
  float vec[4][2][PQ];                         // chunks with the true mask: a wave's copy of cs and dt
};

__device__ __forceinline__ float rdlane(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ __forceinline__ float from_lane(float v, int l) { return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * l, __float_as_int(v))); }
__device__ __forceinline__ void meet() {       // this wave's LDS accesses are done, and then all waves'
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ unsigned pack2(float a, float b) {
  const bf16x2 p = {(bf16_t)a, (bf16_t)b};
  return __builtin_bit_cast(unsigned, p);
}
__device__ __forceinline__ u32x4 times(u32x4 v, const float (&w)[8]) {
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack2(bf16_lo(v[e]) * w[2 * e], bf16_hi(v[e]) * w[2 * e + 1]);
  return o;
}
__device__ __forceinline__ u32x4 times(u32x4 v, float w) {
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = pack2(bf16_lo(v[e]) * w, bf16_hi(v[e]) * w);
  return o;
}

// softplus_fast without branches
__device__ __forceinline__ float softplus_flat(float x) {
  const float e = __expf(x);
  float sp = 0.6931471805599453f * __builtin_amdgcn_logf(1.f + e), near = e - 0.5f * e * e;
  asm("" : "+v"(sp), "+v"(near));
  sp = e < 1e-3f ? near : sp;
  return x > 20.f ? x : sp;
}

template <int PT, bool OUT>
__global__ __launch_bounds__(256, OUT ? 2 : 3) void ssd_par_kernel(ParArgs a) {
  constexpr int NP = PT / 2, ODD = PT & 1, PIECES = 2 * PT, NX = (PIECES + 3) / 4, P = 16 * PT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  typedef ParSmem<PT, OUT> Smem;
  Smem& sm = *reinterpret_cast<Smem*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, kq = lane >> 4, q4 = lc >> 2, p4 = lane & 3;
  // heads of a group on one XCD where there are eight groups: B, C and C.B^T stay in its L2
  const int g = blockIdx.x % a.G, hr = blockIdx.x / a.G, hpg = a.H / a.G, b = blockIdx.y, seg = blockIdx.z;
  const int h = a.group_map ? hr * a.G + g : g * hpg + hr;
  const int L = a.L, c0 = seg * a.seg_chunks, c1 = min(c0 + a.seg_chunks, a.nchunks);
  const int64_t bh = (int64_t)b * a.H + h;
  const unsigned lds0 = lds_addr_of(smem_raw);
  auto tr = [&](unsigned p) { return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4*)(size_t)p); };

  const bf16_t* const xg = a.x + (int64_t)b * a.xsb + h * P;
  const bf16_t* const Bg = a.Bm + (int64_t)b * a.bsb + (int64_t)g * a.bsg + 32 * w;
  const bf16_t* const Cg = OUT ? a.Cm + (int64_t)b * a.csb + (int64_t)g * a.csg : nullptr;
  const bf16_t* const dtg = a.dt + (int64_t)b * a.dsb + h;
  const bf16_t* const cbg = OUT ? a.cb + ((int64_t)b * a.G + g) * a.nchunks * (PFR * 512) + (w < 2 ? w : 2 * w - 2) * 512 : nullptr;
  bf16_t* const yg = OUT ? a.y + (int64_t)b * a.ysb + h * P : nullptr;

  // ---- what a step needs from memory, one step ahead in registers
  const int tq = 16 * w + lc;                              // token of the chunk whose outputs this lane holds
  // piece i of a chunk of x that this thread moves: row << 16 | place in LDS, bit 31: halves exchanged (put_x)
  unsigned xp[NX];
  auto piece_of = [&](int id, int i, int& r, int& c) __attribute__((always_inline)) {
    const int p = min(id + 256 * i, PQ * PIECES - 1);
    r = p / PIECES;
    c = p - r * PIECES;
  };
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    int r, c;
    piece_of(tid, i, r, c);
    const bool single = ODD && c >= 4 * NP;
    const unsigned o = single ? NP * XPAIR + ((r * 32) ^ ((r & 8) << 4)) + (c & 1) * 16 : (c >> 2) * XPAIR + r * 64 + (c & 3) * 16;
    xp[i] = (unsigned)r << 16 | o | (!single && (r & 8) ? 0x80000000u : 0u);
  }
  // Byte offsets from a chunk's first row; rows past the end repeat the last one (finite; dt is 0 there).  Formed for the first chunk and again for a last,
  // partial one: between the loads themselves there is no branch (the compiler would wait for all of them at the next use of one).
  constexpr int NY = (PIECES + 3) / 4, YROW = 32 * PT + 16;    // pieces a lane has of its wave's 16 rows of y; bytes a row in LDS (an odd number of pieces)
  unsigned xo[NX], bo[4], co[OUT ? 4 : 1], yx[OUT ? NY : 1];
  const int xs2 = (int)a.xsl * 2, bs2 = (int)a.bsl * 2, cs2_ = (int)a.csl * 2, ys2 = (int)a.ysl * 2;
  auto offsets = [&](int last) __attribute__((always_inline)) {
    int id = tid;
    asm volatile("" : "+v"(id));                           // (formed here, not kept in registers all the way)
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      int r, c;
      piece_of(id, i, r, c);
      xo[i] = (unsigned)(min(r, last) * xs2 + c * 16);
    }
    const int l = id & 63;
#pragma unroll
    for (int i = 0; i < 4; ++i) bo[i] = (unsigned)(min(16 * i + (l >> 2), last) * bs2 + (l & 3) * 16);
    if constexpr (OUT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) co[i] = (unsigned)(min(16 * w + 4 * i + (l >> 4), last) * cs2_ + (l & 15) * 16);
    }
  };
  auto y_piece = [&](int l, int i, int& r, int& c) __attribute__((always_inline)) {
    const int q = min(l + 64 * i, 16 * PIECES - 1);
    r = q / PIECES;
    c = q - r * PIECES;
  };
  auto offsets_y = [&](int last) __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));
#pragma unroll
    for (int i = 0; i < NY; ++i) {
      int r, c;
      y_piece(l, i, r, c);
      yx[i] = (unsigned)(min(16 * w + r, last) * xs2 + c * 16);
    }
  };
  u32x4 xr[NX], br[4], cr[4], cbr[2];
  unsigned short dr;
  typedef __attribute__((address_space(1))) const unsigned char* gp;
  auto at = [](const bf16_t* base, unsigned off) { return *(__attribute__((address_space(1))) const u32x4*)((gp)base + off); };
  auto load_x = [&](int c) __attribute__((always_inline)) {
    const bf16_t* p = xg + (int64_t)(c * PQ) * a.xsl;
#pragma unroll
    for (int i = 0; i < NX; ++i) xr[i] = at(p, xo[i]);
  };
  // dt of a chunk: 16 tokens a wave (four lanes each)
  auto load_dt = [&](int c) __attribute__((always_inline)) {
    const int t = min(c * PQ + 16 * w + (lane >> 2), L - 1) - c * PQ;
    dr = *(__attribute__((address_space(1))) const unsigned short*)((gp)(dtg + (int64_t)(c * PQ) * a.dsl) + (unsigned)(t * (int)a.dsl * 2));
  };
  auto put_dt = [&](int buf) __attribute__((always_inline)) { sm.dt[buf][16 * w + (lane >> 2)] = bf16_lo(dr); };
  auto load_b = [&](int c) __attribute__((always_inline)) {
    const bf16_t* p = Bg + (int64_t)(c * PQ) * a.bsl;
#pragma unroll
    for (int i = 0; i < 4; ++i) br[i] = at(p, bo[i]);
  };
  auto load_c = [&](int c) __attribute__((always_inline)) {
    const bf16_t* p = Cg + (int64_t)(c * PQ) * a.csl;
#pragma unroll
    for (int i = 0; i < 4; ++i) cr[i] = at(p, co[i]);
  };
  auto load_cb = [&](int c) __attribute__((always_inline)) {   // (waves 0 and 1 have one fragment)
    const bf16_t* p = cbg + (int64_t)c * (PFR * 512);
    cbr[0] = at(p, 16u * lane);
    cbr[1] = at(p + (w < 2 ? 0 : 512), 16u * lane);
  };

  // ---- chunk vectors: lane = token.  weight of x, row factor of y, factor of the state, what brings a raised chunk down again
  const float Ah = a.A[h], bias = a.dt_bias ? a.dt_bias[h] : 0.f;
  float wv = 0.f, rf = 0.f, dec = 0.f, csl = 0.f, decay_sum = 0.f;
  bool up = false, masked = false;
  auto prep = [&](int c, float raw) __attribute__((always_inline)) {
    float d = raw + bias;
    if (a.softplus) d = softplus_flat(d);
    d = c * PQ + lane < L ? fminf(fmaxf(d, a.dt_min), a.dt_max) : 0.f;
    const float cs = wave_incl_scan_dpp(d * Ah), cl = rdlane(cs, 63);
    const float cs2 = cs * LOG2E, cl2 = cl * LOG2E;
    decay_sum += cl;
    if constexpr (!OUT) {
      wv = __builtin_amdgcn_exp2f(cl2 - cs2) * d;
      dec = __builtin_amdgcn_exp2f(cl2);
      return;
    }
    masked = !(-cl2 <= MASK_FROM);
    up = !masked && !(-cl2 <= UP);
    const float k = up ? UP : 0.f;
    wv = masked ? 1.f : __builtin_amdgcn_exp2f(cl2 - cs2 + k) * d;
    rf = __builtin_amdgcn_exp2f(masked ? cs2 : cs2 - cl2 - k);
    dec = __builtin_amdgcn_exp2f(cl2 + k);
    csl = cl2;
    if (masked) {
      sm.vec[w][0][lane] = cs2;
      sm.vec[w][1][lane] = d;
    }
  };
  // x~ into LDS: a pair of tiles in rows of 64 bytes (the 8-byte halves of a piece change places in rows 8 .. 15 mod 16), a single tile in rows of 32
  // (rows r and r ^ 4 change places there): transposing reads meet no bank twice
  auto put_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      u32x4 v = times(xr[i], from_lane(wv, (xp[i] >> 16) & 63));
      if ((int)xp[i] < 0) v = u32x4{v[2], v[3], v[0], v[1]};
      if (256 * i + 255 < PQ * PIECES || tid + 256 * i < PQ * PIECES) *(u32x4*)(&sm.x[buf][xp[i] & 0xffff]) = v;
    }
  };
  const unsigned pr_lo = (8 * kq + q4) * 64 + 16 * p4, sw8 = 8 * (kq & 1);
  auto pair_frag = [&](unsigned base, int half, int ks) {   // 16 columns (half of a pair), tokens 32 ks + 8 kq + 0..7
    const unsigned p = base + pr_lo + ((8 * half) ^ sw8) + ks * 2048;
    return cat4(tr(p), tr(p + 256));
  };
  auto x_frag = [&](unsigned xt, int t, int ks) {
    if (ODD && t == PT - 1) {
      const unsigned p = xt + NP * XPAIR + 256 * kq + 32 * q4 + 8 * p4 + 1024 * ks;
      return cat4(tr(p + 128 * (kq & 1)), tr(p + 128 * ((kq & 1) ^ 1)));
    }
    return pair_frag(xt + (t >> 1) * XPAIR, t & 1, ks);
  };
  auto col_of = [&](int t, int r) { return ODD && t == PT - 1 ? 32 * NP + r : 32 * (t >> 1) + 8 * (r >> 2) + 4 * (t & 1) + (r & 3); };

  // ---- state: X[i][t], lane (lc, kq): rows n = 32 w + 8 kq + 4 i + 0..3, column col_of(t, lc)
  f32x4 X[2][PT];
  auto decayed = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < PT; ++t) { X[0][t] *= dec; X[1][t] *= dec; }
  };
  auto leave = [&](int buf) __attribute__((always_inline)) {
    if (!OUT || !masked) decayed();
    if constexpr (OUT) {
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        const f32x4 u = X[0][t], v = X[1][t];
        *(u32x4*)(&sm.snap[buf][((t * 4 + w) * 64 + lane) * 8]) = u32x4{pack2(u[0], u[1]), pack2(u[2], u[3]), pack2(v[0], v[1]), pack2(v[2], v[3])};
      }
      if (masked) decayed();
    }
  };

  offsets(L - 1 - c0 * PQ);
  if constexpr (OUT) offsets_y(L - 1 - c0 * PQ);
  load_dt(c0);
  const unsigned short dr0 = dr;
  load_dt(min(c0 + 1, c1 - 1));
  load_x(c0);
  load_b(c0);
  if constexpr (OUT) {
    load_c(c0);
    load_cb(c0);
  }
#pragma unroll
  for (int t = 0; t < PT; ++t) X[0][t] = X[1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int LOCW = 2 * PT * 64 * 4;                    // floats of a wave's part of a local state
  const int64_t seg_step = (int64_t)gridDim.y * a.H;
  float before = 0.f;                                      // sums of dt A of the segments in front
  if constexpr (OUT) {
    const float* lp = a.loc + (bh * 4 + w) * LOCW + lane * 4;
    float F = 1.f;
    if (seg > 0) {
      const float sd = lane < seg ? a.segdec[lane * seg_step + bh] : 0.f;
      f32x4 part[2][PT];                                   // (the next segment's part is asked for before this one's is added)
      auto get = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < PT; ++t) part[i][t] = *(const f32x4*)(lp + j * (seg_step * 4 * LOCW) + (i * PT + t) * 256);
      };
      float sum = 0.f;
      get(seg - 1);
      for (int j = seg - 1;; --j) {
        f32x4 now[2][PT];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < PT; ++t) now[i][t] = part[i][t];
        if (j > 0) get(j - 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < PT; ++t) X[i][t] += F * now[i][t];
        sum += rdlane(sd, j);
        F = sum * LOG2E >= FORGOTTEN ? __builtin_amdgcn_exp2f(sum * LOG2E) : 0.f;
        if (j == 0 || F == 0.f) break;
      }
      if (a.total_decay) for (int j = 0; j < seg; ++j) before += rdlane(sd, j);
    }
    if (a.init && F != 0.f) {
#pragma unroll
      for (int t = 0; t < PT; ++t) {
        const float* ip = a.init + (bh * P + col_of(t, lc)) * PN + 32 * w + 8 * kq;
        X[0][t] += F * *(const f32x4*)ip;
        X[1][t] += F * *(const f32x4*)(ip + 4);
      }
    }
  }
  put_dt((c0 + 1) & 1);
  dr = dr0;
  put_dt(c0 & 1);
  meet();
  auto put_c = [&]() __attribute__((always_inline)) {      // rows of 256 bytes, piece p of row r at place p ^ r
    if constexpr (OUT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *(u32x4*)(&sm.b[w][256 * (4 * i + kq) + 16 * (lc ^ (4 * i + kq))]) = cr[i];
    }
  };
  put_c();
  prep(c0, sm.dt[c0 & 1][lane]);
  leave(c0 & 1);
  put_x(c0 & 1);
  meet();

  const float Dh = OUT && a.D ? a.D[h] : 0.f;
  const unsigned xt0 = lds0 + (unsigned)offsetof(Smem, x), bt = lds0 + (unsigned)offsetof(Smem, b) + w * (PQ * 64);
  for (int c = c0; c < c1; ++c) {
    const int buf = c & 1, cn = min(c + 1, c1 - 1);
    const unsigned xt = xt0 + buf * (unsigned)sizeof(sm.x[0]);
    bf16x8 cf[OUT ? 4 : 1];
    if constexpr (OUT) {
#pragma unroll
      for (int q = 0; q < 4; ++q) cf[q] = *(const bf16x8*)(&sm.b[w][256 * lc + 16 * ((4 * q + kq) ^ lc)]);
    }
    // B: this wave's slice, halves of a piece exchanged in rows 8 .. 15 mod 16 (lanes 32 .. 63)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 v = br[i];
      if (lane & 32) v = u32x4{v[2], v[3], v[0], v[1]};
      *(u32x4*)(&sm.b[w][1024 * i + 16 * lane]) = v;
    }
    if ((cn + 1) * PQ > L) offsets(L - 1 - cn * PQ);
    if (OUT && (c + 1) * PQ > L) offsets_y(L - 1 - c * PQ);
    load_b(cn);
    load_x(cn);
    load_dt(min(c + 2, c1 - 1));
    f32x4 yo[PT];
    if constexpr (OUT) {
#pragma unroll
      for (int t = 0; t < PT; ++t) yo[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int t = 0; t < PT; ++t) yo[t] = mfma16(*(const bf16x8*)(&sm.snap[buf][((t * 4 + q) * 64 + lane) * 8]), cf[q], yo[t]);
      load_c(cn);
      if (masked) {                                          // (the outputs from the state: their row factor first)
        const float ct = from_lane(rf, tq);
#pragma unroll
        for (int t = 0; t < PT; ++t) yo[t] *= ct;
      }
    }
    u32x4 rw[NY];                                          // x as it is, for y
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 xf[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) xf[t] = x_frag(xt, t, ks);
      if constexpr (OUT) {
        if (ks == 1) {
#pragma unroll
          for (int i = 0; i < NY; ++i) rw[i] = at(xg + (int64_t)(c * PQ) * a.xsl, yx[i]);
        }
        if (ks == 0 || w >= 2) {
          bf16x8 m = __builtin_bit_cast(bf16x8, cbr[ks]);
          if (masked) {
            const float(&vc)[2][PQ] = sm.vec[w];           // CB[t][s] 2^(cs_t - cs_s) dt_s [s <= t]
            const int s0 = 32 * ks + 8 * kq;
            const float cst = vc[0][tq];
            float f[8];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const f32x4 c4 = *(const f32x4*)&vc[0][s0 + 4 * e], d4 = *(const f32x4*)&vc[1][s0 + 4 * e];
#pragma unroll
              for (int j = 0; j < 4; ++j) f[4 * e + j] = __builtin_amdgcn_exp2f(s0 + 4 * e + j <= tq ? cst - c4[j] : -__builtin_inff()) * d4[j];
            }
            m = __builtin_bit_cast(bf16x8, times(__builtin_bit_cast(u32x4, m), f));
          }
#pragma unroll
          for (int t = 0; t < PT; ++t) yo[t] = mfma16(xf[t], m, yo[t]);
        }
        if (masked) {
          const int s0 = 32 * ks + 8 * kq;
          float f[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) f[j] = __builtin_amdgcn_exp2f(csl - sm.vec[w][0][s0 + j]) * sm.vec[w][1][s0 + j];
#pragma unroll
          for (int t = 0; t < PT; ++t) xf[t] = __builtin_bit_cast(bf16x8, times(__builtin_bit_cast(u32x4, xf[t]), f));
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8 bf = pair_frag(bt, i, ks);
#pragma unroll
        for (int t = 0; t < PT; ++t) X[i][t] = mfma16(bf, xf[t], X[i][t]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (OUT) load_cb(cn);
    if (OUT && up) {
      const float down = __builtin_amdgcn_exp2f(-UP);
#pragma unroll
      for (int t = 0; t < PT; ++t) { X[0][t] *= down; X[1][t] *= down; }
    }
    const float ev = !OUT || masked ? 1.f : from_lane(rf, tq);
    if (c + 1 < c1) {
      prep(c + 1, sm.dt[buf ^ 1][lane]);
      put_dt(buf);
      put_x(buf ^ 1);
      leave(buf ^ 1);
    }
    if constexpr (OUT) {
      // x and y through the wave's tile: whole rows to and from memory, the results' layout in between
      unsigned char* const tile = sm.b[w];
#pragma unroll
      for (int i = 0; i < NY; ++i) {
        int r, cc;
        y_piece(lane, i, r, cc);
        *(u32x4*)(tile + r * YROW + cc * 16) = rw[i];
      }
      unsigned char* const mine = tile + lc * YROW;
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        u32x4* const m = (u32x4*)(mine + 64 * u + 16 * kq);
        const u32x4 x = *m;
        u32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4& s = yo[2 * u + (e >> 1)];
          const int j = 2 * (e & 1);
          v[e] = pack2(fmaf(s[j], ev, Dh * bf16_lo(x[e])), fmaf(s[j + 1], ev, Dh * bf16_hi(x[e])));
        }
        *m = v;
      }
      if (ODD) {
        u32x2* const m = (u32x2*)(mine + 64 * NP + 8 * kq);
        const u32x2 x = *m;
        const f32x4& s = yo[PT - 1];
        *m = u32x2{pack2(fmaf(s[0], ev, Dh * bf16_lo(x[0])), fmaf(s[1], ev, Dh * bf16_hi(x[0]))),
                   pack2(fmaf(s[2], ev, Dh * bf16_lo(x[1])), fmaf(s[3], ev, Dh * bf16_hi(x[1])))};
      }
      bf16_t* const yp = yg + (int64_t)(c * PQ + 16 * w) * a.ysl;
#pragma unroll
      for (int i = 0; i < NY; ++i) {
        int r, cc;
        y_piece(lane, i, r, cc);
        const u32x4 v = *(const u32x4*)(tile + r * YROW + cc * 16);
        if (c * PQ + 16 * w + r < L && (64 * i + 63 < 16 * PIECES || lane + 64 * i < 16 * PIECES))
          *(u32x4*)((unsigned char*)yp + (unsigned)(r * ys2 + cc * 16)) = v;
      }
    }
    if (c + 1 < c1) {
      put_c();
      meet();
    }
  }
  if constexpr (OUT) {
    if (seg == a.nseg - 1) {
      if (a.final_state) {
#pragma unroll
        for (int t = 0; t < PT; ++t) {
          float* fp = a.final_state + (bh * P + col_of(t, lc)) * PN + 32 * w + 8 * kq;
          *(f32x4*)fp = X[0][t];
          *(f32x4*)(fp + 4) = X[1][t];
        }
      }
      if (a.total_decay && tid == 0) a.total_decay[bh] = before + decay_sum;
    }
  } else {
    float* lp = a.loc + ((seg * seg_step + bh) * 4 + w) * LOCW + lane * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < PT; ++t) *(f32x4*)(lp + (i * PT + t) * 256) = X[i][t];
    if (tid == 0) a.segdec[seg * seg_step + bh] = decay_sum;
  }
}

template <int PT>
hipError_t launch_par(const ParArgs& a, int batch, hipStream_t st) {
  typedef ParSmem<PT, true> So;
  typedef ParSmem<PT, false> Sl;
  static_assert(2 * sizeof(So) <= 160 * 1024 && 3 * sizeof(Sl) <= 160 * 1024, "LDS budget");
  static const hipError_t attr = hipFuncSetAttribute((const void*)ssd_par_kernel<PT, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(So));
  if (attr != hipSuccess) return attr;
  if (a.nseg > 1) ssd_par_kernel<PT, false><<<dim3(a.H, batch, a.nseg - 1), 256, sizeof(Sl), st>>>(a);
  ssd_par_kernel<PT, true><<<dim3(a.H, batch, a.nseg), 256, sizeof(So), st>>>(a);
  return hipSuccess;
}

}  // namespace

// bytes of the local states and the decays of `nseg` segments
size_t tv_ssd_par_workspace_bytes(int batch, int nheads, int headdim, int nseg) {
  return nseg > 1 ? (size_t)(nseg - 1) * batch * nheads * (headdim * PN + 1) * sizeof(float) : 0;
}

// the caller has checked alignments and 32-bit offsets (tv_ssd_head_supported); headdim 32, 64 or 80, nseg <= 64
int tv_ssd_par_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* cb, const void* D,
                      const void* dt_bias, const void* init_state, void* y, void* final_state, void* total_decay, int batch, int seqlen, int nheads,
                      int headdim, int ngroups, int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg,
                      int64_t csb, int64_t csl, int64_t csg, int64_t ysb, int64_t ysl, int dt_softplus, float dt_min, float dt_max, int group_map,
                      int nseg, int seg_chunks, void* workspace, hipStream_t st) {
  ParArgs a;
  a.x = (const bf16_t*)x; a.dt = (const bf16_t*)dt; a.Bm = (const bf16_t*)Bm; a.Cm = (const bf16_t*)Cm; a.cb = (const bf16_t*)cb;
  a.A = (const float*)A; a.D = (const float*)D; a.dt_bias = (const float*)dt_bias; a.init = (const float*)init_state;
  a.y = (bf16_t*)y; a.final_state = (float*)final_state; a.total_decay = (float*)total_decay;
  a.loc = (float*)workspace;
  a.segdec = (float*)workspace + (size_t)(nseg - 1) * batch * nheads * headdim * PN;
  a.L = seqlen; a.H = nheads; a.G = ngroups; a.nchunks = (seqlen + PQ - 1) / PQ; a.nseg = nseg; a.seg_chunks = seg_chunks;
  a.xsb = xsb; a.xsl = xsl; a.dsb = dsb; a.dsl = dsl; a.bsb = bsb; a.bsl = bsl; a.bsg = bsg; a.csb = csb; a.csl = csl; a.csg = csg;
  a.ysb = ysb; a.ysl = ysl;
  a.softplus = dt_softplus; a.group_map = group_map; a.dt_min = dt_min; a.dt_max = dt_max;
  hipError_t e = headdim == 80 ? launch_par<5>(a, batch, st) : headdim == 64 ? launch_par<4>(a, batch, st) : launch_par<2>(a, batch, st);
  if (e != hipSuccess) {
    tv_set_error("ssd_par: %s", hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  TV_LAUNCH_CHECK();
}
