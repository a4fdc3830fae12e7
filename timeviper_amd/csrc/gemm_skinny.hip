// Products of a few rows with a weight matrix, y[m][n] = sum_k x[m][k] W[n][k], 2 <= m <= 32: one decoded token for each of several
// sequences.  Every weight byte is used once, for at most 32 rows: HBM-bound (N K 2 bytes).
//
// The matrix-vector kernels (gemv.hip) hold f(x) in LDS and spend a dot-product instruction per 2 weights and row of x: at four rows
// the vector pipe is what a work-group waits for, and above four rows there was only the library, whose 32 x 16 tiles read the
// weights at 2 - 4 TB/s.  Here the products run on the matrix cores (v_mfma_f32_16x16x32_bf16, W rows on the A side, so that a lane's 4 accumulator
// registers are 4 consecutive outputs of one row of x), which makes their cost independent of the number of rows up to 16, and
// what is left is a stream of W:
//   * a work-group owns `rw` <= 32 rows of W and its waves split K; the partial sums meet once, in LDS, behind the loop.  Inside
//     it there is no barrier: W and x both arrive by LDS-DMA in a ring PRIVATE to the wave (a stage is 64 columns: 8 rows x 128
//     bytes an instruction), NS - 1 stages ahead of the math behind counted vmcnt waits.  x (a few hundred KiB) comes from L2.
//   * `rw` is not a multiple of a tile: it is chosen so that all work-groups run at once and carry the same number of bytes (rows of
//     a tile past `rw` repeat the last one: the matrix pipe has the time, the memory does not see them).
// fp32 accumulation, one rounding of y.
// Measured (weights not in any cache; library or matrix-vector kernel before -> here): 22 656 x 4 480, 12 rows 66 -> 32.0 us (6.3 TB/s), 4 rows
// 42.8 -> 30.9; 4 480 x 15 680, 12 rows 43.5 -> 25.0, 4 rows 45.0 -> 22.7; 2 048 x 7 680, 4 rows 13.2 -> 7.4 (latency: 31 MB); 17 to 32 rows are
// level with the library at the largest sizes (22 656 x 4 480, 32 rows: 40.6 and 40.5) and up to 1.6 times as fast below (52 -> 34 at
// 4 480 x 15 680): there x from L2 is as many bytes as W.
#include "gemm_skinny.hpp"

namespace {
using namespace ssdk;

enum { SK_BF16 = 0, SK_F32 = 1, SK_ADD = 2, SK_RELU2 = 3, SK_PAIR = 4, SK_CONV = 5 };
constexpr int SK_KC = 64;                          // columns of a stage

struct SkArgs {
  const bf16_t *x, *x2, *W, *bias;
  bf16_t *y, *h_out, *act;
  float *y32, *res_out;
  const float* res;
  int epi, round;                                  // round: SK_F32 of the bf16 rounding
  int M, N, K, rw;                                 // rw: rows of W per work-group (SK_PAIR, second part: gate rows per work-group)
  int64_t xs, x2s, ldw, ys, as;
  int n1, ff, wg1, rw1;                            // SK_PAIR: work-groups [0, wg1) take rw1 rows each of the first n1
  bf16_t* conv_state;                              // SK_CONV: outputs [conv_lo, conv_hi) pass a width-4 causal-conv update + SiLU
  const bf16_t *conv_w, *conv_b;
  int conv_lo, conv_hi;
  const bf16_t* u;                                 // GLU: y = gelu_tanh(bf16(.)) * row u_ids[m] (NULL: m) of u
  const int64_t* u_ids;
  int64_t us, u_rows;
};

// WI, XI: copy instructions (8 rows each) per stage of W and of x; NW waves; NS ring stages a wave
// GLU: the gate of a layer's token side (128 outputs a token) with the row that meets it, which waits for the token's id and then for a row of
// the table: both are asked for beside the ring's first stages, .5 us.  Gate and projection 2 048 wide: 8 rows, a launch between the two products, 9.3 -> 7.8 us; 4
// rows, in front of every work-group of the second one, 8.7 -> 7.6.
template <int WI, int XI, int NW, int NS, bool GLU>
__global__ __launch_bounds__(NW * 64) void skinny_stream_kernel(SkArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char sk_smem[];
  constexpr int NT = (WI + 1) / 2, MT = XI == 4 ? 2 : 1, T = NT * MT;
  constexpr int STAGE = (WI + XI) * 1024, OPS = WI + XI;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;

  // rows of this work-group: LDS row r holds row row_of(r) of W
  const bool two = a.epi == SK_PAIR, pair = two && (int)blockIdx.x >= a.wg1;       // (work-group uniform, as are all branches on epi)
  const int rw = two && !pair ? a.rw1 : a.rw;
  const int n0 = ((int)blockIdx.x - (pair ? a.wg1 : 0)) * rw;
  const int rows = min(rw, (two ? (pair ? a.ff : a.n1) : a.N) - n0);             // (>= 1: launcher)
  const bf16_t* x = pair ? a.x2 : a.x;
  const int64_t xs = pair ? a.x2s : a.xs;
  const bf16_t* Wb = a.W + (int64_t)(pair ? a.n1 + n0 : n0) * a.ldw;

  // ---- copies: instruction i, lane l -> LDS row 8 i + l / 8, 16-byte chunk l % 8, which holds source chunk (l % 8) ^ ((row >> 1) & 7)
  unsigned vw[WI], vx[XI];
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int row = 8 * i + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    int64_t r;
    if (pair) r = row < 4 * WI ? min(row, rows - 1) : (int64_t)a.ff + min(row - 4 * WI, rows - 1);      // gate rows | up rows
    else r = min(row, rows - 1);
    vw[i] = (unsigned)((r * a.ldw + ch * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int row = 8 * i + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    vx[i] = (unsigned)(((int64_t)min(row, a.M - 1) * xs + ch * 8) * 2);
  }
  const unsigned ring = lds_addr_of(sk_smem) + (unsigned)(wave * NS * STAGE);
  // ---- this wave's share of the K / 64 stages
  const int nst = a.K / SK_KC;
  const int s0 = (int)((int64_t)nst * wave / NW), ns = (int)((int64_t)nst * (wave + 1) / NW) - s0;
  auto issue = [&](int i, int S) __attribute__((always_inline)) {
    const unsigned dst = ring + (unsigned)(S * STAGE);
    glds_rows<WI, true>(uniform_ptr(Wb + (int64_t)(s0 + i) * SK_KC), vw, dst);
    glds_rows<XI, false>(uniform_ptr(x + (int64_t)(s0 + i) * SK_KC), vx, dst + WI * 1024);
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef __attribute__((address_space(3))) const bf16x8 lds_bf16x8;
  // fragment reads: row n of a 16-row tile, 16-byte chunk 4 ks + g  (an odd last tile reads 8 rows past the rows of W: outputs nobody stores)
  const unsigned f0 = (unsigned)(n * 128 + ((g ^ (n >> 1)) << 4)), f1 = f0 ^ 64u;
  auto compute = [&](int S) __attribute__((always_inline)) {
    const unsigned st = ring + (unsigned)(S * STAGE);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const unsigned f = st + (ks ? f1 : f0);
      bf16x8 xf[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) xf[m] = *(lds_bf16x8*)(size_t)(f + (unsigned)(WI * 1024 + m * 2048));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8 wf = *(lds_bf16x8*)(size_t)(f + (unsigned)(t * 2048));
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = mfma16(wf, xf[m], acc[t][m]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (the next copies overwrite an older stage: every read of it is back)
  };
  // GLU: this thread's outputs (a work-group has at most NW * 64 quads of them: one pass of the epilogue's loop)
  bf16_t uv[4] = {};
  int64_t ur = 0;
  if constexpr (GLU) {
    const int m = tid < 2 * WI * a.M ? tid % a.M : 0;
    ur = a.u_ids ? a.u_ids[m] : m;
  }
#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (j < ns) issue(j, j);
  if constexpr (GLU) {
    const bool ok = ur >= 0 && ur < a.u_rows;                 // (callers check ids on the host; a bad one counts as zeros)
    const int q = tid < 2 * WI * a.M ? tid / a.M : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uv[j] = a.u[(ok ? ur : 0) * a.us + n0 + min(4 * q + j, rows - 1)];
      if (!ok) uv[j] = (bf16_t)0.f;
    }
  }
  int S = 0, i = 0;
  for (; i + NS - 1 < ns; ++i) {
    issue(i + NS - 1, S == 0 ? NS - 1 : S - 1);               // the stage that step i - 1 has left
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OPS * (NS - 1)) : "memory");
    compute(S);
    S = S == NS - 1 ? 0 : S + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  for (; i < ns; ++i) {
    compute(S);
    S = S == NS - 1 ? 0 : S + 1;
  }

  // ---- the waves meet: [wave][tile][lane] f32x4 over the ring, which every wave has left
  __syncthreads();
  f32x4* part = (f32x4*)sk_smem;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) part[(wave * T + t * MT + m) * 64 + lane] = acc[t][m];
  __syncthreads();
  // 4 consecutive outputs (quad q) of row m of x
  auto total = [&](int q, int m) __attribute__((always_inline)) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) s += part[(w * T + (q >> 2) * MT + (m >> 4)) * 64 + (q & 3) * 16 + (m & 15)];
    return s;
  };
  const int nq = pair ? WI : 2 * WI;
  for (int e = tid; e < nq * a.M; e += NW * 64) {
    const int q = e / a.M, m = e - q * a.M;
    if (4 * q >= rows) continue;
    f32x4 s = total(q, m);
    if (pair) {
      const f32x4 u = total(q + WI, m);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * q + j < rows) {
          const int o = n0 + 4 * q + j;
          a.act[(int64_t)m * a.as + o] = (bf16_t)(gelu_tanh_f(s[j] + (float)a.bias[o]) * (u[j] + (float)a.bias[a.ff + o]));
        }
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * q + j < rows) {
        const int o = n0 + 4 * q + j;
        float v = s[j];
        if (!two && a.bias) v += (float)a.bias[o];
        if (a.epi == SK_F32) a.y32[(int64_t)m * a.ys + o] = a.round ? (float)(bf16_t)v : v;
        else if (a.epi == SK_ADD) {
          v += a.res[(int64_t)m * a.N + o];
          a.res_out[(int64_t)m * a.N + o] = v;
          if (a.h_out) a.h_out[(int64_t)m * a.N + o] = (bf16_t)v;
        } else {
          bf16_t out = (bf16_t)v;
          if constexpr (GLU) out = (bf16_t)(gelu_tanh_f((float)out) * (float)uv[j]);
          if (a.epi == SK_RELU2) {                            // squared ReLU of what the product would have written
            const float r = fmaxf((float)out, 0.f);
            out = (bf16_t)(r * r);
          }
          if (a.epi == SK_CONV && o >= a.conv_lo && o < a.conv_hi) {
            // tv_causal_conv1d_update on this channel: window = state[1..3], out
            const int c = o - a.conv_lo;
            bf16_t* st = a.conv_state + ((int64_t)m * (a.conv_hi - a.conv_lo) + c) * 4;
            const bf16x4 old = *(const bf16x4*)st, wv = *(const bf16x4*)(a.conv_w + (int64_t)c * 4);
            const bf16x4 win = {old[1], old[2], old[3], out};
            float ac = a.conv_b ? (float)a.conv_b[c] : 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t) ac = fmaf((float)wv[t], (float)win[t], ac);
            *(bf16x4*)st = win;
            out = (bf16_t)silu_f(ac);
          }
          a.y[(int64_t)m * a.ys + o] = out;
        }
      }
  }
}

template <int WI, int XI, int NW, int NS, bool GLU = false>
int launch_one(const SkArgs& a, int wgs, hipStream_t st) {
  constexpr int T = ((WI + 1) / 2) * (XI == 4 ? 2 : 1);
  constexpr int RING = NW * NS * (WI + XI) * 1024, PART = NW * T * 1024;
  constexpr int LDS = (RING > PART ? RING : PART) + 1024;       // (+ 1 KiB: the tile reads past 8-row operands)
  static_assert(LDS <= 160 * 1024, "ring");
  static const hipError_t attr = hipFuncSetAttribute((const void*)skinny_stream_kernel<WI, XI, NW, NS, GLU>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (attr != hipSuccess) {
    tv_set_error("gemm_rows: cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  skinny_stream_kernel<WI, XI, NW, NS, GLU><<<dim3((unsigned)wgs), NW * 64, LDS, st>>>(a);
  TV_LAUNCH_CHECK();
}

// The ring: about 32 - 48 KiB of W in flight per compute unit.  One work-group per compute unit: 8 waves of 3 stages (2 048 x 7 680, four
// rows: 7.4 us against 8.2 with 4 waves of 4); several: 4 waves of 3, two work-groups resident (15 680 x 4 480, 12 rows: 22.9 us; 24.0 with 4
// stages, 27 with 8 waves).  More than 16 rows of x: 2 stages, the x tile takes the room.
template <int XI>
int launch_xi(const SkArgs& a, int wi, int wgs, bool one, hipStream_t st) {
  constexpr int NS = XI == 4 ? 2 : 3;
#define SK_GO(WI) case WI: return one ? launch_one<WI, XI, 8, NS>(a, wgs, st) : launch_one<WI, XI, 4, NS>(a, wgs, st)
  switch (wi) { SK_GO(1); SK_GO(2); SK_GO(3); default: break; }
  return one ? launch_one<4, XI, 8, NS>(a, wgs, st) : launch_one<4, XI, 4, NS>(a, wgs, st);
#undef SK_GO
}

// Rows of W per work-group: the fewest rounds of one work-group per compute unit whose share is at most 32 rows, all shares alike
// (4 480 rows: 18 in 249 work-groups; 9 in 498 read x twice as often, 24.0 against 22.7 us at K = 15 680).
int rows_share(int64_t n, bool& one) {
  const int cus = tv_cu_count();
  const int64_t rounds = (n + 32ll * cus - 1) / (32ll * cus);
  one = rounds == 1;
  return (int)((n + rounds * cus - 1) / (rounds * cus));
}

}  // namespace

bool tv_skinny_takes(const void* x, const void* W, int M, int K, int64_t xs, int64_t ldw, int64_t far_rows) {
  // (copies are 16 bytes a lane at 32-bit offsets from a work-group's first row; a stage is 64 columns)
  return M >= 2 && M <= TV_GEMM_ROWS_MAX && K >= SK_KC && K % SK_KC == 0 && xs % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x & 15) == 0 &&
         ((uintptr_t)W & 15) == 0 && xs >= 0 && ldw >= 0 && 32 * xs * 2 < (1ll << 31) && (far_rows + 32) * ldw * 2 < (1ll << 31);
}

static int skinny_go(SkArgs& a, hipStream_t st) {
  bool one;
  int wgs, wi;
  if (a.epi == SK_PAIR) {
    const int r = (rows_share((int64_t)a.n1 + 2ll * a.ff, one) + 1) & ~1;       // (<= 32)
    a.rw1 = r;
    a.rw = r / 2;
    a.wg1 = (a.n1 + r - 1) / r;
    wgs = a.wg1 + (a.ff + a.rw - 1) / a.rw;
    wi = (r + 7) / 8;
  } else {
    a.rw = rows_share(a.N, one);
    wgs = (a.N + a.rw - 1) / a.rw;
    wi = (a.rw + 7) / 8;
  }
  if (a.M <= 8) return launch_xi<1>(a, wi, wgs, one, st);
  if (a.M <= 16) return launch_xi<2>(a, wi, wgs, one, st);
  return launch_xi<4>(a, wi, wgs, one, st);
}

// the matrix-vector entry points hand products of two to four rows without a prologue over (gemv.hip)
int tv_skinny_add(const void* x, const void* W, const void* bias, const float* residual, float* residual_out, void* h_out, int M, int N, int K,
                  int64_t xs, int64_t ldw, hipStream_t st) {
  SkArgs a{};
  a.x = (const bf16_t*)x; a.W = (const bf16_t*)W; a.bias = (const bf16_t*)bias; a.res = residual; a.res_out = residual_out;
  a.h_out = (bf16_t*)h_out; a.epi = SK_ADD; a.M = M; a.N = N; a.K = K; a.xs = xs; a.ldw = ldw;
  return skinny_go(a, st);
}

int tv_skinny_pair(const void* x, const void* x2, const void* W, const void* bias, void* y, void* act, int M, int n1, int ff, int K,
                   int64_t xs, int64_t x2s, int64_t ldw, int64_t ys, int64_t as, hipStream_t st) {
  SkArgs a{};
  a.x = (const bf16_t*)x; a.x2 = (const bf16_t*)x2; a.W = (const bf16_t*)W; a.bias = (const bf16_t*)bias; a.y = (bf16_t*)y; a.act = (bf16_t*)act;
  a.M = M; a.N = n1; a.K = K; a.xs = xs; a.x2s = x2s; a.ldw = ldw; a.ys = ys; a.as = as; a.n1 = n1; a.ff = ff;
  a.epi = ff ? SK_PAIR : SK_BF16;
  if (!ff) a.bias = nullptr;
  return skinny_go(a, st);
}

extern "C" int tv_gemm_rows_fwd(const void* x, const void* W, const void* bias, void* y, int y_dtype, int M, int N, int K, int64_t x_stride,
                                int64_t ldw, int64_t y_stride, int epilogue, void* conv_state, const void* conv_weight, const void* conv_bias,
                                int conv_row0, int conv_channels, void* stream) {
  TV_CHECK_ARG(x && W && y, "gemm_rows: null pointer");
  TV_CHECK_ARG(M >= 2 && M <= TV_GEMM_ROWS_MAX && N >= 1 && K >= 1, "gemm_rows: M %d must be 2..%d, N %d and K %d positive", M, TV_GEMM_ROWS_MAX, N, K);
  TV_CHECK_ARG(y_dtype == TV_BF16 || (y_dtype == TV_F32 && (epilogue == 0 || epilogue == TV_GEMM_ROWS_ROUND) && !conv_state), "gemm_rows: y dtype %d", y_dtype);
  TV_CHECK_ARG(epilogue == 0 || (epilogue == TV_GEMM_ROWS_RELU2 && !conv_state) || (epilogue == TV_GEMM_ROWS_ROUND && y_dtype == TV_F32), "gemm_rows: epilogue %d", epilogue);
  if (!tv_skinny_takes(x, W, M, K, x_stride, ldw, 0))
    TV_UNSUPPORTED("gemm_rows: K must be a multiple of %d, the row strides of x and W of 8 elements, x and W 16-byte aligned", SK_KC);
  SkArgs a{};
  a.x = (const bf16_t*)x; a.W = (const bf16_t*)W; a.bias = (const bf16_t*)bias;
  if (y_dtype == TV_F32) a.y32 = (float*)y; else a.y = (bf16_t*)y;
  a.M = M; a.N = N; a.K = K; a.xs = x_stride; a.ldw = ldw; a.ys = y_stride;
  a.round = epilogue == TV_GEMM_ROWS_ROUND;
  a.epi = y_dtype == TV_F32 ? SK_F32 : epilogue == TV_GEMM_ROWS_RELU2 ? SK_RELU2 : SK_BF16;
  if (conv_state) {
    TV_CHECK_ARG(conv_weight && conv_row0 >= 0 && conv_channels > 0 && conv_row0 + conv_channels <= N,
                 "gemm_rows: conv epilogue rows [%d, %d) outside the %d outputs", conv_row0, conv_row0 + conv_channels, N);
    if (((uintptr_t)conv_state & 7) || ((uintptr_t)conv_weight & 7)) TV_UNSUPPORTED("gemm_rows: conv state / weight must be 8-byte aligned");
    a.epi = SK_CONV;
    a.conv_state = (bf16_t*)conv_state; a.conv_w = (const bf16_t*)conv_weight; a.conv_b = (const bf16_t*)conv_bias;
    a.conv_lo = conv_row0; a.conv_hi = conv_row0 + conv_channels;
  }
  return skinny_go(a, (hipStream_t)stream);
}

extern "C" int tv_gemm_rows_add_fwd(const void* x, const void* W, const void* bias, const float* residual, float* residual_out, void* h_out, int M,
                                    int N, int K, int64_t x_stride, int64_t ldw, void* stream) {
  TV_CHECK_ARG(x && W && residual && residual_out, "gemm_rows_add: null pointer");
  TV_CHECK_ARG(M >= 2 && M <= TV_GEMM_ROWS_MAX && N >= 1 && K >= 1, "gemm_rows_add: M %d must be 2..%d, N %d and K %d positive", M, TV_GEMM_ROWS_MAX, N, K);
  if (!tv_skinny_takes(x, W, M, K, x_stride, ldw, 0))
    TV_UNSUPPORTED("gemm_rows_add: K must be a multiple of %d, the row strides of 8 elements, x and W 16-byte aligned", SK_KC);
  return tv_skinny_add(x, W, bias, residual, residual_out, h_out, M, N, K, x_stride, ldw, (hipStream_t)stream);
}

extern "C" int tv_gemm_rows_pair_fwd(const void* x, const void* x2, const void* W, const void* bias, void* y, void* act, int M, int n1, int ff,
                                     int K, int64_t x_stride, int64_t x2_stride, int64_t ldw, int64_t y_stride, int64_t act_stride, void* stream) {
  TV_CHECK_ARG(x && W && y && (ff == 0 || (x2 && bias && act)), "gemm_rows_pair: null pointer");
  TV_CHECK_ARG(M >= 2 && M <= TV_GEMM_ROWS_MAX && n1 >= 1 && ff >= 0 && K >= 1, "gemm_rows_pair: M %d must be 2..%d, rows %d + 2 x %d, K %d positive", M,
               TV_GEMM_ROWS_MAX, n1, ff, K);
  if (!tv_skinny_takes(x, W, M, K, x_stride, ldw, ff) || (ff && !tv_skinny_takes(x2, W, M, K, x2_stride, ldw, ff)))
    TV_UNSUPPORTED("gemm_rows_pair: K must be a multiple of %d, the row strides of 8 elements, operands 16-byte aligned", SK_KC);
  return tv_skinny_pair(x, x2, W, bias, y, act, M, n1, ff, K, x_stride, x2_stride, ldw, y_stride, act_stride, (hipStream_t)stream);
}

extern "C" int tv_gemm_rows_glu_fwd(const void* x, const void* W, const void* u, const int64_t* u_ids, int64_t u_rows, void* y, int M, int N, int K,
                                    int64_t x_stride, int64_t ldw, int64_t u_stride, int64_t y_stride, void* stream) {
  TV_CHECK_ARG(x && W && u && y, "gemm_rows_glu: null pointer");
  TV_CHECK_ARG(M >= 2 && M <= TV_GEMM_ROWS_MAX && N >= 1 && K >= 1 && u_rows >= (u_ids ? 1 : M),
               "gemm_rows_glu: M %d must be 2..%d, N %d and K %d positive, %lld rows of u", M, TV_GEMM_ROWS_MAX, N, K, (long long)u_rows);
  if (!tv_skinny_takes(x, W, M, K, x_stride, ldw, 0))
    TV_UNSUPPORTED("gemm_rows_glu: K must be a multiple of %d, the row strides of x and W of 8 elements, x and W 16-byte aligned", SK_KC);
  SkArgs a{};
  a.x = (const bf16_t*)x; a.W = (const bf16_t*)W; a.y = (bf16_t*)y; a.M = M; a.N = N; a.K = K; a.xs = x_stride; a.ldw = ldw; a.ys = y_stride;
  a.u = (const bf16_t*)u; a.u_ids = u_ids; a.u_rows = u_rows; a.us = u_stride;
  a.epi = SK_BF16;
  bool one;
  a.rw = rows_share(N, one);
  if (a.rw > 8) TV_UNSUPPORTED("gemm_rows_glu: %d outputs, at most 8 a compute unit", N);
  const int wgs = (N + a.rw - 1) / a.rw;
  hipStream_t st = (hipStream_t)stream;
  if (M <= 8) return launch_one<1, 1, 8, 3, true>(a, wgs, st);
  if (M <= 16) return launch_one<1, 2, 8, 3, true>(a, wgs, st);
  return launch_one<1, 4, 8, 2, true>(a, wgs, st);
}
