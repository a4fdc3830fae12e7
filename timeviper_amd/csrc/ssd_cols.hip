// S3 for short sequences: the recurrence of ssd_head.hip with a 16-COLUMN SLICE of a head per group of waves.
//
// A head's 80 (64, 32) columns of x, y and the state never meet in the recurrence: y[t][p] and S[p][:] need x[t][p] alone beside dt, B and
// C.  With a wave per head a prompt of a few thousand tokens leaves 128 waves on 1 024 SIMDs, each taking 5 us a step; cutting the
// sequence into segments instead (what long sequences do) costs the chain of the segments' states and a second pass over y, 30 -
// 60 us.  Here a work-group takes 4 slices that follow each other in a B / C group (128 bytes of every x and y row), and the chain of
// latencies that is then left of a step — dt -> softplus -> prefix sum -> weights -> x~ -> products -> y, 2.6 us as one wave's
// program — is cut into three that run side by side, a wave each per slice (one of each on every SIMD):
//   vectors  copies a step ahead (LDS-DMA, two stages), and prep(k + 1): the chunk's decays, frame, weights and mode
//   state    X' (= 0 or X') += B^T x~ of chunk k; leaves the bf16 copy of the state that ENTERS chunk k + 1 in LDS
//   output   Yoff (from that copy) + Ydiag of chunk k, row factors, D x; y through LDS, so that whole 128-byte lines are stored
//            (32 bytes a row straight from the registers are partial lines)
// Two barriers a step: k's inputs are complete | last readers of the two buffers with one copy (state copy, y tile) are done.
// Arithmetic, frames and modes are ssd_head.hip's (floating frame, reset and standard steps; see there); a standard step takes its
// mask factors one by one.
// Up to 7 chunks come here, 9 at head dim 80, 24 where the heads are too many for more than three segments (use_cols in ssd_head.hip); beyond, the chain is cut (ssd_par.hip).
// What is left is instruction issue — three waves a SIMD with about 350 vector and 38 matrix instructions a step, 1.6 us — and, in heads that
// decay by more than 2^199 a chunk, the mask factors of a standard step (2.6 us).
// Two stages, not three: the copies of the step ahead have the step's 2 us, and a call waits for one chunk before its first step instead of two (three | two, 128 heads x 80, fresh
// Mamba-2 decays and decays of a hundredth: 150 tokens 14.8 | 14.4, 10.4 | 9.8 us; 250: 21.0 | 20.7, 12.2 | 11.4; 500: 29.5 | 28.8, 18.7 | 17.5; one chunk level).
// Measured (128 heads x 80, 8 groups, whole operator, against a wave per head): 203 tokens 35 -> 17 us, 390: 46 -> 19.
#include "ssd_common.hpp"

namespace {
using namespace ssdk;

constexpr int HQ = 64, HN = 128, CP = 16;      // tokens a chunk, d_state, columns a slice
constexpr int NFR = 6;                         // causal fragments of C.B^T of a chunk, 512 elements each
constexpr float RMAX = 100.f, RESET_THR = 64.f;

struct ColsArgs {
  const bf16_t *x, *dt, *Bm, *Cm, *cb;
  const float *A, *D, *dt_bias, *init;
  bf16_t* y;
  float *final_state, *total_decay;
  int L, H, G, sub, nchunks;                   // sub: slices a head
  int64_t xsb, xsl, dsb, dsl, bsb, bsl, bsg, csb, csl, csg, ysb, ysl;
  int softplus, group_map;
  float dt_min, dt_max;
};

struct __attribute__((aligned(16))) ColVec {   // a chunk's vectors of a slice's head, by token
  float yw[HQ];       // weight of x in Ydiag (the frame Yoff is formed in); standard steps: 2^(cs_e - cs_t) dt_t, e the last of the 16-token tile
  float sw[HQ];       // weight of x in the state update; standard steps: dt
  float ecs[HQ];      // row factor 2^(cs_t + E)
  float cs[HQ];       // inclusive prefix sum of dt A, times log2(e)
};
struct __attribute__((aligned(16))) ColStage {
  bf16_t bt[HQ * HN], ct[HQ * HN];
  unsigned dt[4][64];                          // of the chunk behind
};
struct __attribute__((aligned(16))) ColSmem {
  ColStage st[2];
  bf16_t xr[2][4][HQ * CP];
  bf16_t yt[4][HQ * CP];
  bf16_t snap[4][4 * 64 * 8];                  // [slice][quarter of the state rows][lane] 16 bytes: Yoff's operand
  ColVec v[2][4];
  int mode[2][4];                              // shift of the frame | reset << 16 | standard << 17
  float e_end[4];
};

typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4v;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float rdlane(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
// this wave's LDS accesses are done, and then all waves'
__device__ __forceinline__ void meet() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// x fragment (element j = token 32 ks + 8 kq + j) times w[32 ks + 8 kq + j], rounded to bf16
__device__ __forceinline__ bf16x8 scaled(bf16x8 f, const float* w) {
  const u32x4v u = __builtin_bit_cast(u32x4v, f);
  const f32x4 w0 = *(const f32x4*)w, w1 = *(const f32x4*)(w + 4);
  u32x4v o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bf16x2 pk = {(bf16_t)(bf16_lo(u[e]) * (e < 2 ? w0[2 * e] : w1[2 * e - 4])), (bf16_t)(bf16_hi(u[e]) * (e < 2 ? w0[2 * e + 1] : w1[2 * e - 3]))};
    o[e] = __builtin_bit_cast(unsigned, pk);
  }
  return __builtin_bit_cast(bf16x8, o);
}

__global__ __launch_bounds__(768) void ssd_cols_kernel(ColsArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  ColSmem& sm = *reinterpret_cast<ColSmem*>(smem_raw);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int w = wave & 3, role = wave >> 2;                    // slice of the work-group; 0 vectors, 1 state, 2 output
  const int lc = lane & 15, kq = lane >> 4, q4 = (lane & 15) >> 2, p4 = lane & 3;
  const int b = blockIdx.y, hpg = a.H / a.G;
  const int g = blockIdx.x % a.G;
  const int sl = (blockIdx.x / a.G) * 4 + w;                   // slice within the group
  const int hr = sl / a.sub;
  const int h = a.group_map ? (hr * a.G + g) : (g * hpg + hr);
  const int col = (h * a.sub + (sl - hr * a.sub)) * CP;        // first column of x and y, first row of the state
  const int L = a.L, nchunks = a.nchunks;
  const unsigned lds0 = lds_addr_of(smem_raw);
  constexpr int XROW = 2 * CP;
  typedef __attribute__((address_space(3))) const bf16x8 lds8;
  auto tr = [&](unsigned p) { return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4*)(size_t)p); };
  const unsigned xr_lo = (8 * kq + q4) * XROW + 8 * p4;
  auto x_tile = [&](int S) { return lds0 + (unsigned)offsetof(ColSmem, xr) + (unsigned)S * 8192u + 2048u * w; };
  auto x_frag = [&](unsigned xt, int ks) { return cat4(tr(xt + xr_lo + ks * (32 * XROW)), tr(xt + xr_lo + ks * (32 * XROW) + 4 * XROW)); };

  if (role == 0) {
    // ------------------------------------------------------------------ copies and vectors
    const bf16_t* Bg = a.Bm + (int64_t)b * a.bsb + (int64_t)g * a.bsg;
    const bf16_t* Cg = a.Cm + (int64_t)b * a.csb + (int64_t)g * a.csg;
    const bf16_t* xg = a.x + (int64_t)b * a.xsb + col;
    const bf16_t* dtg = a.dt + (int64_t)b * a.dsb + (h & ~1);  // the dword that holds this head's dt
    const bool odd = (h & 1) != 0;
    const int l4 = lane >> 4, l16 = lane & 15;
    // Whole chunks: lane offsets from the chunk's first row, formed once (piece k of a group of four: + its rows - 1024 k, the
    // instruction offset moves both addresses).  B and C: 4 rows of 256 bytes a piece, B chunk ^ 4 (row & 3), C chunk ^ (row & 15).
    unsigned ob[4], oc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = 16 * w + 4 * k + l4;
      ob[k] = (unsigned)((row * a.bsl + (l16 ^ (4 * (row & 3))) * 8) * 2) - 1024u * k;
      oc[k] = (unsigned)((row * a.csl + (l16 ^ (row & 15)) * 8) * 2) - 1024u * k;
    }
    const unsigned ox0 = (unsigned)(((lane >> 1) * a.xsl + (lane & 1) * 8) * 2), ox1 = ox0 + (unsigned)(64 * a.xsl) - 1024u;
    const unsigned dB = lds0 + (unsigned)offsetof(ColStage, bt) + 4096u * w, dC = lds0 + (unsigned)offsetof(ColStage, ct) + 4096u * w;
    const unsigned dD = lds0 + (unsigned)offsetof(ColStage, dt) + 256u * w;
    // stage of chunk c, and dt of chunk c + 1
    auto issue = [&](int c, int S) __attribute__((always_inline)) {
      const unsigned so = (unsigned)S * (unsigned)sizeof(ColStage), dX = x_tile(S);
      const int t0 = c * HQ, last = L - 1 - t0;
      const void* bp = uniform_ptr(Bg + (int64_t)t0 * a.bsl);
      const void* cp = uniform_ptr(Cg + (int64_t)t0 * a.csl);
      const void* xp = uniform_ptr(xg + (int64_t)t0 * a.xsl);
      if (last >= HQ - 1) {
        unsigned keep;
        glds16x4(bp, ob[0], ob[1], ob[2], ob[3], dB + so);
        glds16x4(cp, oc[0], oc[1], oc[2], oc[3], dC + so);
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\t"
                     "global_load_lds_dwordx4 %2, %3 offset:1024\n\ts_mov_b32 m0, %0"
                     : "=&s"(keep) : "v"(ox0), "v"(ox1), "s"(xp), "s"(dX) : "memory");
      } else {                                                 // the last, partial chunk: rows past the end repeat the last one (finite)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int row = 16 * w + 4 * k + l4, rr = min(row, last);
          glds16(bp, (unsigned)((rr * a.bsl + (l16 ^ (4 * (row & 3))) * 8) * 2), dB + so + 1024u * k);
          glds16(cp, (unsigned)((rr * a.csl + (l16 ^ (row & 15)) * 8) * 2), dC + so + 1024u * k);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
          glds16(xp, (unsigned)((min(32 * k + (lane >> 1), last) * a.xsl + (lane & 1) * 8) * 2), dX + 1024u * k);
      }
      const int t1 = min(t0 + HQ, L - 1);
      glds4(uniform_ptr(dtg + (int64_t)t1 * a.dsl), (unsigned)(min(lane, L - 1 - t1) * a.dsl * 2), dD + so);
    };
    const float Ah = a.A[h], bias = a.dt_bias ? a.dt_bias[h] : 0.f;
    float decay_total = 0.f, E = 0.f;
    // vectors and mode of chunk c (decisions and arithmetic of ssd_head_kernel's prep)
    auto prep = [&](int c, int S, float raw) __attribute__((always_inline)) {
      ColVec& vec = sm.v[S][w];
      float d = 0.f;
      if (c * HQ + lane < L) {
        d = raw + bias;
        if (a.softplus) d = softplus_fast(d);
        d = fminf(fmaxf(d, a.dt_min), a.dt_max);
      }
      const float cs = wave_incl_scan_dpp(d * Ah);
      const float cl = rdlane(cs, 63);
      const float cs2 = cs * 1.4426950408889634f, cl2 = cl * 1.4426950408889634f;
      const int mode = -(E + cl2) <= RMAX ? 0 : -cl2 <= 2.f * RMAX - 1.f ? 1 : 2;
      const float mshift = mode == 1 ? __builtin_floorf(RMAX - E) : 0.f;
      const float Euse = E + mshift;
      const bool std_ = mode == 2, rst = !std_ && cl2 <= -RESET_THR;
      const float p0 = rdlane(cs2, 15), p1 = rdlane(cs2, 31), p2 = rdlane(cs2, 47);
      const float ce = lane < 16 ? p0 : lane < 32 ? p1 : lane < 48 ? p2 : cl2;
      const float fw = __builtin_amdgcn_exp2f(std_ ? ce - cs2 : -cs2 - Euse) * d;
      vec.yw[lane] = fw;
      vec.sw[lane] = std_ ? d : rst ? __builtin_amdgcn_exp2f(cl2 - cs2 - RMAX) * d : fw;
      vec.ecs[lane] = __builtin_amdgcn_exp2f(cs2 + Euse);
      vec.cs[lane] = cs2;
      decay_total += cl;
      E = std_ ? 0.f : rst ? RMAX : Euse + cl2;
      if (lane == 0) sm.mode[S][w] = ((int)-mshift & 0xffff) | (rst || std_ ? 1 << 16 : 0) | (std_ ? 1 << 17 : 0);
    };
    auto dt_of = [&](int S) __attribute__((always_inline)) {
      const unsigned raw = sm.st[S].dt[w][lane];
      return odd ? bf16_hi(raw) : bf16_lo(raw);
    };
    float r0 = (float)dtg[(int64_t)min(lane, L - 1) * a.dsl + (odd ? 1 : 0)];
    asm volatile("" : "+v"(r0));                               // (from here on only copies are counted; as a copy among the others it comes later: 100 tokens 10.1, so 10.5)
    issue(0, 0);
    prep(0, 0, r0);
    meet();                                                    // (the state wave reads chunk 0's mode)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int S = 0;
    for (int k = 0; k < nchunks; ++k) {
      meet();
      if (k + 1 < nchunks) {
        issue(k + 1, S ^ 1);                                   // (the stage that step k - 1 has left)
        prep(k + 1, S ^ 1, dt_of(S));
      } else if (lane == 0) {
        sm.e_end[w] = E;
      }
      meet();
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // (in front of the next meeting)
      S ^= 1;
    }
    if (a.total_decay && lane == 0 && sl == hr * a.sub) a.total_decay[(int64_t)b * a.H + h] = decay_total;
    meet();
  } else if (role == 1) {
    // ------------------------------------------------------------------ state: tile i, lane (lc, kq): S[p = lc][n = 32 (i >> 1) + 8 kq + 4 (i & 1) + 0..3] 2^-E
    f32x4 X[8];
    const int64_t srow = ((int64_t)b * a.H * a.sub * CP + col + lc) * HN + 8 * kq;
#pragma unroll
    for (int i = 0; i < 8; ++i) X[i] = a.init ? *(const f32x4*)(a.init + srow + 32 * (i >> 1) + 4 * (i & 1)) : f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned bsw = q4 << 6, b_lo = (8 * kq + q4) * 256 + p4 * 16;
    // y: this wave stores rows 16 w .. + 15 of a chunk, of all four slices: lane = row lane / 8, 16-byte piece lane % 8
    const int ys_sl = sl - w + ((lane & 7) >> 1), ys_hr = ys_sl / a.sub, ys_h = a.group_map ? (ys_hr * a.G + g) : (g * hpg + ys_hr);
    bf16_t* const yg = a.y + (int64_t)b * a.ysb + (int64_t)(16 * w + (lane >> 3)) * a.ysl + (ys_h * a.sub + (ys_sl - ys_hr * a.sub)) * CP + (lane & 1) * 8;
    const bf16_t* yrd = &sm.yt[(lane & 7) >> 1][(16 * w + (lane >> 3)) * CP + (lane & 1) * 8];
    auto store_y = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8 v = *(const bf16x8*)(yrd + i * 8 * CP);
        const int t = c * HQ + 8 * i;
        if (t + 16 * w + (lane >> 3) < L) *(bf16x8*)(yg + (int64_t)t * a.ysl) = v;
      }
    };
    auto leave = [&]() __attribute__((always_inline)) {        // the bf16 copy of the state rows n = 32 q + 8 kq + 0..7: an MFMA operand
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x8 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          o[j] = (bf16_t)X[2 * q][j];
          o[4 + j] = (bf16_t)X[2 * q + 1][j];
        }
        *(bf16x8*)(&sm.snap[w][(q * 64 + lane) * 8]) = o;
      }
    };
    auto to_frame = [&](int mode) __attribute__((always_inline)) {
      const int shift = (int)(short)(mode & 0xffff);
      if (!shift) return;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) X[i][j] = __builtin_amdgcn_ldexpf(X[i][j], shift);
    };
    meet();
    to_frame(__builtin_amdgcn_readfirstlane(sm.mode[0][w]));
    leave();
    int S = 0;
    for (int k = 0; k < nchunks; ++k) {
      meet();
      const unsigned Bt = lds0 + (unsigned)S * (unsigned)sizeof(ColStage) + (unsigned)offsetof(ColStage, bt), xt = x_tile(S);
      const int md = __builtin_amdgcn_readfirstlane(sm.mode[S][w]);
      if (k > 0) store_y(k - 1);                               // (here, where nothing waits for memory)
      bf16x8 x0 = x_frag(xt, 0), x1 = x_frag(xt, 1);
      if (md & (1 << 17)) {
        const ColVec& vec = sm.v[S][w];
        const float cl2 = vec.cs[HQ - 1];
        float f0[8], f1[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          f0[j] = __builtin_amdgcn_exp2f(cl2 - vec.cs[8 * kq + j]) * vec.sw[8 * kq + j];
          f1[j] = __builtin_amdgcn_exp2f(cl2 - vec.cs[32 + 8 * kq + j]) * vec.sw[32 + 8 * kq + j];
        }
        x0 = scaled(x0, f0);
        x1 = scaled(x1, f1);
      } else {
        x0 = scaled(x0, &sm.v[S][w].sw[8 * kq]);
        x1 = scaled(x1, &sm.v[S][w].sw[32 + 8 * kq]);
      }
      if (md & (1 << 16)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) X[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned bp = Bt + ((bsw ^ (64u * (i >> 1))) + b_lo) + (i & 1) * 8;
        X[i] = mfma16(cat4(tr(bp), tr(bp + 1024)), x0, X[i]);
        X[i] = mfma16(cat4(tr(bp + 8192), tr(bp + 9216)), x1, X[i]);
      }
      meet();
      if (k + 1 < nchunks) {
        to_frame(__builtin_amdgcn_readfirstlane(sm.mode[S ^ 1][w]));      // the next chunk's frame
        leave();
      }
      S ^= 1;
    }
    meet();
    store_y(nchunks - 1);
    if (a.final_state) {
      const float sc = __builtin_amdgcn_exp2f(sm.e_end[w]);
#pragma unroll
      for (int i = 0; i < 8; ++i) *(f32x4*)(a.final_state + srow + 32 * (i >> 1) + 4 * (i & 1)) = X[i] * sc;
    }
  } else {
    // ------------------------------------------------------------------ output
    const float Dh = a.D ? a.D[h] : 0.f;
    const bf16_t* cbg = a.cb + ((int64_t)b * a.G + g) * a.nchunks * (NFR * 512) + lane * 8;
    const unsigned c_lo = lc * 256, c_z = (kq ^ lc) << 4, xv_lo = lc * XROW + 8 * kq;
    // C.B^T fragments straight into registers, two steps ahead: two sets that take turns (a copy from one to the other would wait for it)
    bf16x8 cb0[NFR], cb1[NFR];
    auto load_cb = [&](bf16x8 (&c)[NFR], int k) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < NFR; ++f) c[f] = *(const bf16x8*)(cbg + (int64_t)min(k, nchunks - 1) * (NFR * 512) + f * 512);
    };
    load_cb(cb0, 0);
    load_cb(cb1, 1);
    meet();
    int S = 0;
    auto step = [&](int k, bf16x8 (&cbv)[NFR]) __attribute__((always_inline)) {
      meet();
      const unsigned Ct = lds0 + (unsigned)S * (unsigned)sizeof(ColStage) + (unsigned)offsetof(ColStage, ct), xt = x_tile(S);
      const ColVec& vec = sm.v[S][w];
      const bool standard = (__builtin_amdgcn_readfirstlane(sm.mode[S][w]) & (1 << 17)) != 0;
      f32x4 yo[4];
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) yo[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bf16x8 sb = *(const bf16x8*)(&sm.snap[w][(q * 64 + lane) * 8]);
        const unsigned cp = Ct + ((c_z ^ (64u * q)) + c_lo);
#pragma unroll
        for (int ti = 0; ti < 4; ++ti) yo[ti] = mfma16(sb, *(lds8*)(size_t)(cp + ti * 4096), yo[ti]);
        if (q & 1) __builtin_amdgcn_sched_barrier(0);          // (all sixteen operands at once do not fit the registers)
      }
      bf16x8 xw[2] = {x_frag(xt, 0), x_frag(xt, 1)};
      float ev[4];
      u32x2 xr[4];
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) {
        ev[ti] = vec.ecs[16 * ti + lc];
        typedef __attribute__((address_space(3))) const u32x2 lds_u32x2;
        xr[ti] = *(lds_u32x2*)(size_t)(xt + xv_lo + ti * (16 * XROW));
      }
      // Ydiag on top of Yoff: the A operand is x~, the B operand the causal C.B^T fragment
      if (!standard) {
        xw[0] = scaled(xw[0], &vec.yw[8 * kq]);
        xw[1] = scaled(xw[1], &vec.yw[32 + 8 * kq]);
#pragma unroll
        for (int f = 0; f < NFR; ++f) {
          const int ti = f == 0 ? 0 : f == 1 ? 1 : f < 4 ? 2 : 3;
          yo[ti] = mfma16(xw[f == 3 || f == 5], cbv[f], yo[ti]);
        }
      } else {
        // true-mask form: row factors now, CB .* 2^(cs_t - cs_s) dt_s [s <= t] in place of C.B^T, raw x
#pragma unroll
        for (int ti = 0; ti < 4; ++ti) {
          yo[ti] *= ev[ti];
          ev[ti] = 1.f;
        }
#pragma unroll
        for (int f = 0; f < NFR; ++f) {
          // the lane's 8 tokens s0 .. + 7 lie in one 16-token tile: in front of t's tile one factor for all of them, in it one each
          const int ti = f == 0 ? 0 : f == 1 ? 1 : f < 4 ? 2 : 3, s0 = (f == 3 || f == 5 ? 32 : 0) + 8 * kq, t = 16 * ti + lc;
          const float ct = vec.cs[t], u = __builtin_amdgcn_exp2f(fminf(ct - vec.cs[s0 | 15], 0.f));
          const bool own = (s0 >> 4) == ti, may_own = f != 2 && f != 4;
          bf16x8 m;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float fac = (s0 >> 4) < ti ? u * vec.yw[s0 + j] : 0.f;
            if (may_own) {
              const float e = __builtin_amdgcn_exp2f(s0 + j <= t ? ct - vec.cs[s0 + j] : -__builtin_inff()) * vec.sw[s0 + j];
              fac = own ? e : fac;
            }
            m[j] = (bf16_t)((float)cbv[f][j] * fac);
          }
          yo[ti] = mfma16(xw[f == 3 || f == 5], m, yo[ti]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      load_cb(cbv, k + 2);
      // the lane holds columns 4 kq + 0..3 of token 16 ti + lc
      u32x2 yv[4];
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) {
        const bf16x2 p0 = {(bf16_t)fmaf(yo[ti][0], ev[ti], Dh * bf16_lo(xr[ti][0])), (bf16_t)fmaf(yo[ti][1], ev[ti], Dh * bf16_hi(xr[ti][0]))};
        const bf16x2 p1 = {(bf16_t)fmaf(yo[ti][2], ev[ti], Dh * bf16_lo(xr[ti][1])), (bf16_t)fmaf(yo[ti][3], ev[ti], Dh * bf16_hi(xr[ti][1]))};
        yv[ti] = u32x2{__builtin_bit_cast(unsigned, p0), __builtin_bit_cast(unsigned, p1)};
      }
      meet();
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) *(u32x2*)(&sm.yt[w][(16 * ti + lc) * CP + 4 * kq]) = yv[ti];
      S ^= 1;
    };
    for (int k = 0; k < nchunks; k += 2) {
      step(k, cb0);
      if (k + 1 < nchunks) step(k + 1, cb1);
    }
    meet();
  }
}

}  // namespace

// the caller has checked alignments and 32-bit offsets (tv_ssd_head_supported)
int tv_ssd_cols_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* cb, const void* D,
                       const void* dt_bias, const void* init_state, void* y, void* final_state, void* total_decay, int batch, int seqlen, int nheads,
                       int headdim, int ngroups, int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg,
                       int64_t csb, int64_t csl, int64_t csg, int64_t ysb, int64_t ysl, int dt_softplus, float dt_min, float dt_max, int group_map,
                       hipStream_t st) {
  ColsArgs a;
  a.x = (const bf16_t*)x; a.dt = (const bf16_t*)dt; a.Bm = (const bf16_t*)Bm; a.Cm = (const bf16_t*)Cm; a.cb = (const bf16_t*)cb;
  a.A = (const float*)A; a.D = (const float*)D; a.dt_bias = (const float*)dt_bias; a.init = (const float*)init_state;
  a.y = (bf16_t*)y; a.final_state = (float*)final_state; a.total_decay = (float*)total_decay;
  a.L = seqlen; a.H = nheads; a.G = ngroups; a.sub = headdim / CP; a.nchunks = (seqlen + HQ - 1) / HQ;
  a.xsb = xsb; a.xsl = xsl; a.dsb = dsb; a.dsl = dsl; a.bsb = bsb; a.bsl = bsl; a.bsg = bsg; a.csb = csb; a.csl = csl; a.csg = csg;
  a.ysb = ysb; a.ysl = ysl;
  a.softplus = dt_softplus; a.group_map = group_map; a.dt_min = dt_min; a.dt_max = dt_max;
  static_assert(sizeof(ColSmem) <= 160 * 1024, "LDS budget");
  static const hipError_t attr = hipFuncSetAttribute((const void*)ssd_cols_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(ColSmem));
  if (attr != hipSuccess) {
    tv_set_error("ssd_cols: cannot reserve %zu bytes of LDS: %s", sizeof(ColSmem), hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  ssd_cols_kernel<<<dim3(ngroups * (nheads / ngroups * a.sub / 4), batch), 768, sizeof(ColSmem), st>>>(a);
  TV_LAUNCH_CHECK();
}
