// bf16 products of a few hundred to a few thousand rows, C = epilogue(A W^T), on small tiles: 128 x 128, 64 x 128 or 64 x 64 outputs a work-group of eight waves.
//
// gemm.hip's 256 x 256 tiles are a quarter of a round there, and each takes its whole contraction (729 rows: 42 - 51 tiles, 26 us however short it is).  Small tiles
// fill the compute units; the tile is the largest that still gives the chip a round (kernels.small_tile).
//   * Two waves share a quarter of the tile, each with one 32-column half of every stage of 64: a SIMD has two waves, one's products run beside the other's reads and
//     copies, and together they read no more of LDS than one wave would.  The pair meets over the ring behind the loop.  (With four waves, one a SIMD, a stage of a 128 x 128
//     tile was 525 ns even where every copy hit the same lines; 465 with reads and copies dealt out between the products; now 325.  Its 64 KB of fragment reads and 32 of
//     copies take 320 at 128 bytes a clock: LDS bounds it.)
//   * Both operands arrive by LDS-DMA (8 rows x 128 bytes an instruction, 16-byte pieces exchanged on the source side so that fragment reads meet no bank twice) in a ring of
//     NS stages behind counted waits, one barrier a stage.  Four stages: the fragments of stage t + 1 are read during the products of stage t, whose slot, held in registers by
//     then, is filled again (asked for one stage later instead, 1 152 x 4 352 on 64 x 64 tiles takes 19.2 us in place of 16.7).
//   * A stage is a 128-byte piece of each row of W, which memory delivers late where it is not in a cache: in long contractions of 192 rows and more, and in two rounds of tiles, the
//     work-groups together ask for all of W once, a line a lane, beside the first stages (asks_ahead).
//   * Two stages (64 KB): two work-groups a compute unit, for tiles between one round and two (5 120 x 2 048, 1 024 rows: 30.3 us, four stages in two rounds 31.6).
//   * v_mfma_f32_16x16x32_bf16 with W on the A side: two tiles of rows joined by v_permlane16_swap are 16-byte stores, as gemm.hip;
//   * EPI_PART: work-groups share a tile's contraction, their sums meet in a second launch that adds the bias and the residual stream (2 048 x 7 680, us, 256 x 256 tiles in 16 shares ->
//     here: 64 rows 22.5 -> 17.3, 256: 32.8 -> 23.0, 512: 39.2 -> 31.3; 1 024 x 5 120, 256 rows: 27.7 -> 13.9, the library's product and its pass 15.4): fewer sums go through memory.
//   * EPI_GLU: half of a tile's rows of W are those of the gate, half those of the factor N rows further down: a lane holds both of an output.
// fp32 sums, one rounding; the GELU is that of the rounded sum (what the library's product would have written).
// Measured (us on the device, weights out of cache, library | four waves before -> here): 729 x 3 456 x 1 152 17.9 | 15.0 -> 14.0, 729 x 1 152 x 1 152 12.5 | 9.1 -> 8.0, 729 x 1 152 x 4 352
// 22.3 | 26.2 -> 17.9, 1 458 30.7 | 31.2 -> 26.2, 2 916 42.0 | 44.7 -> 34.1, 729 x 5 120 x 2 048 25.9 | 24.8 -> 23.3, 1 458 x 3 456 x 1 152 19.3 | 23.6 -> 23.8.  SigLIP so400m, whole forwards: 1 frame
// of 729 tokens 2.42 -> 2.14 ms, 2: 3.14 -> 2.88, 4: 4.54 -> 4.29.
#include "gemm_common.hpp"

namespace tvgemm {
namespace {

typedef __attribute__((address_space(3))) const bf16x8 lds_bf16x8;

constexpr int GS_THREADS = 512, TOUCH = 4;       // TOUCH: lines of W a thread asks for at most
constexpr int EPI_PART = 6;                      // fp32 sums of a split of the contraction, to a.part [split][M][N]

// WM, WN: a wave's 16-row tiles of A and of W
template <int WM, int WN, int NS, int EPI>
__global__ __launch_bounds__(GS_THREADS, NS == 4 ? 2 : 4) void gemm_small_kernel(GemmArgs a) {
  constexpr int TM = 32 * WM, TN = 32 * WN, STAGE = (TM + TN) * 128, PA = TM / 8, PW = (TM + TN) / 64;
  constexpr bool GLU = EPI == EPI_GLU;
  constexpr int TO = GLU ? TN / 2 : TN;                    // outputs a tile
  extern __shared__ __attribute__((aligned(16))) unsigned char gs_smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = (wave & 3) >> 1, wc = wave & 1, kg = wave >> 2, lc = lane & 15, kq = lane >> 4;

  // ---- tile: ids of an XCD (id % 8) walk neighbouring tiles, bands of group_m tiles of rows
  int id = blockIdx.x, split = 0;
  {
    const int nt = a.tiles_m * a.tiles_n * (EPI == EPI_PART ? a.splits : 1), q = nt / 8, r = nt % 8, x = id % 8;
    id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + id / 8;
  }
  if constexpr (EPI == EPI_PART) {                         // (the splits one after the other: neighbours share columns of both operands)
    split = __builtin_amdgcn_readfirstlane(id / (a.tiles_m * a.tiles_n));
    id -= split * (a.tiles_m * a.tiles_n);
  }
  const int band = id / (a.group_m * a.tiles_n), in_band = id % (a.group_m * a.tiles_n), rows_in_band = min(a.group_m, a.tiles_m - band * a.group_m);
  const int m0 = (band * a.group_m + in_band % rows_in_band) * TM, n0 = in_band / rows_in_band * TO;

  // ---- copies: this wave's pieces of a stage, the rows of A first.  Rows past the end repeat the last one (never stored)
  const unsigned lds0 = lds_addr_of(gs_smem);
  const bf16_t* src[PW];
  unsigned off[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int pc = wave * PW + i;
    const bool isA = pc < PA;
    const int row = 8 * (isA ? pc : pc - PA) + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    int64_t r;
    if (isA) r = min(row, a.M - 1 - m0);
    else if (GLU) r = row < TO ? min(row, a.N - 1 - n0) : (int64_t)a.N + min(row - TO, a.N - 1 - n0);
    else r = min(row, a.N - 1 - n0);
    src[i] = (const bf16_t*)uniform_ptr(isA ? a.A + (int64_t)m0 * a.lda : a.W + (int64_t)n0 * a.ldw);
    off[i] = (unsigned)((r * (isA ? a.lda : a.ldw) + ch * 8) * 2);
  }
  const int all_kt = a.K / BK, kt0 = EPI == EPI_PART ? (int)((int64_t)all_kt * split / a.splits) : 0;
  const int nkt = EPI == EPI_PART ? (int)((int64_t)all_kt * (split + 1) / a.splits) - kt0 : all_kt;
  if constexpr (EPI == EPI_PART) {
#pragma unroll
    for (int i = 0; i < PW; ++i) src[i] = (const bf16_t*)uniform_ptr(src[i] + (int64_t)kt0 * BK);
  }
  auto issue = [&](int t, int S) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PW; ++i) glds16(uniform_ptr(src[i] + t * BK), off[i], lds0 + (unsigned)(S * STAGE + (wave * PW + i) * 1024));
  };

  f32x4 acc[WM][WN];
#pragma unroll
  for (int m = 0; m < WM; ++m)
#pragma unroll
    for (int n = 0; n < WN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned frag = lds0 + (unsigned)(lc * 128 + ((kq ^ (lc >> 1)) << 4));
  const unsigned fa = frag + (unsigned)(wr * WM * 2048), fw = frag + (unsigned)(TM * 128);
  // row of the tile's rows of W at which a wave's tile n starts
  auto w_row = [&](int n) __attribute__((always_inline)) {
    return GLU ? (n < WN / 2 ? 0 : TO) + 16 * (wc * (WN / 2) + n % (WN / 2)) : 16 * (wc * WN + n);
  };
#pragma unroll
  for (int j = 0; j < NS - 1; ++j)
    if (j < nkt) issue(j, j);
  // W on its way from memory, in order, a line a lane, by all work-groups together (the last line again where there is no other)
  float seen[TOUCH] = {};
  if (a.ahead) {
    const int64_t all = (int64_t)gridDim.x * GS_THREADS, pieces = (int64_t)(GLU ? 2 : 1) * a.N * all_kt, most = pieces < 0x7fffffff ? pieces : 0x7fffffff;
#pragma unroll
    for (int i = 0; i < TOUCH; ++i) {
      const int p = (int)min((int64_t)blockIdx.x * GS_THREADS + tid + i * all, most - 1), row = p / all_kt;
      seen[i] = *(const float*)(a.W + (int64_t)row * a.ldw + (p - row * all_kt) * BK);
    }
  }
  bf16x8 af[2][WM], wf[2][WN];                             // by the parity of the stage
  const unsigned fak = fa ^ (unsigned)(kg * 64), fwk = fw ^ (unsigned)(kg * 64);
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  auto read = [&](int i, unsigned st, auto BT) __attribute__((always_inline)) {
    constexpr int B = decltype(BT)::value;
    if (i < WM) af[B][i] = *(lds_bf16x8*)(size_t)(fak + st + (unsigned)(i * 2048));
    else wf[B][i - WM] = *(lds_bf16x8*)(size_t)(fwk + st + (unsigned)(w_row(i - WM) * 128));
  };
  auto products = [&](int lo, int hi, auto BT) __attribute__((always_inline)) {
    constexpr int B = decltype(BT)::value;
#pragma unroll
    for (int i = lo; i < hi; ++i) acc[i / WN][i % WN] = mfma16(wf[B][i % WN], af[B][i / WN], acc[i / WN][i % WN]);
  };
  if constexpr (NS < 4) {
    int S = 0;
    for (int t = 0; t < nkt; ++t) {
      if (t + NS - 2 < nkt) GEMM_WAIT_VM(PW * (NS - 2));
      else GEMM_WAIT_VM(0);
      __builtin_amdgcn_s_barrier();                        // stage t is there for all waves, and all have read stage t - 1
      asm volatile("" ::: "memory");
      if (t + NS - 1 < nkt) issue(t + NS - 1, S == 0 ? NS - 1 : S - 1);
#pragma unroll
      for (int i = 0; i < WM + WN; ++i) read(i, (unsigned)(S * STAGE), I0{});
      products(0, WM * WN, I0{});
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      S = S == NS - 1 ? 0 : S + 1;
    }
  } else {
    // the fragments of stage t + 1 are read, and stage t + NS asked for, between the products of stage t; the wait and the barrier of a step are for the
    // stage behind
    constexpr int MF = WM * WN, HEAD = MF / 4, RD = (WM + WN) / PW;
    int S = 0;                                             // slot of stage t
    auto step = [&](int t, auto BT, auto LASTT) __attribute__((always_inline)) {
      constexpr int B = decltype(BT)::value;
      constexpr bool LAST = decltype(LASTT)::value;        // one of the last steps: the copies run out
      const int S1 = S == NS - 1 ? 0 : S + 1;
      products(0, HEAD, BT);
      __builtin_amdgcn_sched_barrier(0);
      if (!LAST || t + 1 < nkt) {
        if (!LAST || t + NS - 1 < nkt) GEMM_WAIT_VM(PW * (NS - 2));
        else GEMM_WAIT_VM(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                      // stage t + 1 is there for all waves, and all have read stage t, whose slot is filled next
        asm volatile("" ::: "memory");
        const unsigned st = (unsigned)(S1 * STAGE), dst = lds0 + (unsigned)(S * STAGE + wave * PW * 1024);
        const bool more = !LAST || t + NS < nkt;
#pragma unroll
        for (int c = 0; c < PW; ++c) {
          if (more) glds16(src[c] + (t + NS) * BK, off[c], dst + c * 1024);
#pragma unroll
          for (int i = RD * c; i < RD * (c + 1); ++i) read(i, st, std::integral_constant<int, B ^ 1>{});
          products(HEAD + c * (MF - HEAD) / PW, HEAD + (c + 1) * (MF - HEAD) / PW, BT);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        products(HEAD, MF, BT);
      }
      S = S1;
    };
    if (NS - 1 < nkt) {
      issue(NS - 1, NS - 1);
      GEMM_WAIT_VM(PW * (NS - 1));
    } else {
      GEMM_WAIT_VM(0);
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < WM + WN; ++i) read(i, 0u, I0{});
    int t = 0;
    for (; t + NS + 1 < nkt; t += 2) {
      step(t, I0{}, std::false_type{});
      step(t + 1, I1{}, std::false_type{});
    }
    for (; t < nkt; t += 2) {
      step(t, I0{}, std::true_type{});
      if (t + 1 < nkt) step(t + 1, I1{}, std::true_type{});
    }
  }

#pragma unroll
  for (int i = 0; i < TOUCH; ++i) asm volatile("" ::"v"(seen[i]));
  // ---- the two waves of a quarter meet over the ring: each keeps half of the rows, or the first one all of them
  constexpr int KM = WM < 4 ? WM : WM / 2;                 // 16-row tiles a wave keeps
  int mk = wr * WM;                                        // its first one
  f32x4* const meet = (f32x4*)gs_smem;
  auto at = [&](int w, int i) __attribute__((always_inline)) { return meet + (w * (KM * WN) + i) * 64 + lane; };
  static_assert((KM < WM ? 8 : 4) * KM * WN * 1024 <= NS * STAGE, "the meeting fits the ring");
  __syncthreads();
  if constexpr (KM < WM) {
#pragma unroll
    for (int i = 0; i < KM * WN; ++i) {
      const f32x4 lo = acc[i / WN][i % WN], hi = acc[KM + i / WN][i % WN];
      *at(wave ^ 4, i) = kg ? lo : hi;
      acc[i / WN][i % WN] = kg ? hi : lo;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < KM * WN; ++i) acc[i / WN][i % WN] += *at(wave, i);
    mk += kg * KM;
  } else {
    if (kg) {
#pragma unroll
      for (int i = 0; i < WM * WN; ++i) *at(wave ^ 4, i) = acc[i / WN][i % WN];
    }
    __syncthreads();
    if (kg) return;
#pragma unroll
    for (int i = 0; i < WM * WN; ++i) acc[i / WN][i % WN] += *at(wave, i);
  }

  // ---- epilogue: a lane holds, of two joined tiles of rows, 8 columns 16 n + 8 (kq >> 1) .. of row 16 (m + (kq & 1)) + lc
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4e __attribute__((ext_vector_type(4)));
  constexpr int NO = GLU ? WN / 2 : WN;
#pragma unroll
  for (int n = 0; n < NO; ++n) {
    const int col = n0 + 16 * (wc * NO + n) + 8 * (kq >> 1);
    float bv[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, bu[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (EPI != EPI_ACCUM && EPI != EPI_PART && a.bias && col < a.N) {         // (N is a multiple of 8)
      if (a.bias_f32) {
        const f32x4 b0 = *(const f32x4*)((const float*)a.bias + col), b1 = *(const f32x4*)((const float*)a.bias + col + 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) { bv[r] = b0[r]; bv[4 + r] = b1[r]; }
      } else {
        const bf16x8 b8 = *(const bf16x8*)((const bf16_t*)a.bias + col);
#pragma unroll
        for (int r = 0; r < 8; ++r) bv[r] = (float)b8[r];
        if (GLU) {
          const bf16x8 u8 = *(const bf16x8*)((const bf16_t*)a.bias + a.N + col);
#pragma unroll
          for (int r = 0; r < 8; ++r) bu[r] = (float)u8[r];
        }
      }
    }
#pragma unroll
    for (int mp = 0; mp < KM; mp += 2) {
      float v[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[mp][n][r]), __float_as_uint(acc[mp + 1][n][r]), false, false);
        v[r] = __uint_as_float(sw[0]) + bv[r];
        v[4 + r] = __uint_as_float(sw[1]) + bv[4 + r];
        if constexpr (GLU) {
          const auto su = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[mp][n + NO][r]), __float_as_uint(acc[mp + 1][n + NO][r]), false, false);
          v[r] = gelu_tanh_f(v[r]) * (__uint_as_float(su[0]) + bu[r]);
          v[4 + r] = gelu_tanh_f(v[4 + r]) * (__uint_as_float(su[1]) + bu[4 + r]);
        }
      }
      const int row = m0 + 16 * (mk + mp + (kq & 1)) + lc;
      if (row >= a.M || col >= a.N) continue;
      if constexpr (EPI == EPI_PART) {
        float* pp = a.part + ((int64_t)split * a.M + row) * a.N + col;
        *(f32x4*)pp = f32x4{v[0], v[1], v[2], v[3]};
        *(f32x4*)(pp + 4) = f32x4{v[4], v[5], v[6], v[7]};
        continue;
      }
      bf16_t* cp = a.C + (int64_t)row * a.ldc + col;
      if (EPI == EPI_ACCUM) {
        const bf16x8 c8 = *(const bf16x8*)cp;
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] += (float)c8[r];
      }
      if (EPI == EPI_BIAS_GELU) {
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = gelu_erf_f((float)(bf16_t)v[r]);
      }
      u32x4e o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bf16x2 pk = {(bf16_t)v[2 * r], (bf16_t)v[2 * r + 1]};
        o[r] = __builtin_bit_cast(unsigned, pk);
      }
      *(u32x4e*)cp = o;
    }
  }
}

// res_out = res + (sum of the splits, in their order, + bias), C its bf16 copy; four neighbouring outputs a thread
__global__ __launch_bounds__(256) void gemm_small_sum_kernel(GemmArgs a) {
  const int64_t all = (int64_t)a.M * a.N, at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= all) return;
  const f32x4 r = *(const f32x4*)(a.res + at);
  const int col = (int)(at % a.N);
  bf16x4 b = {};
  if (a.bias) b = *(const bf16x4*)((const bf16_t*)a.bias + col);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < a.splits; j += 8) {                  // (a split that is not there repeats the last one and is not added)
    f32x4 t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = *(const f32x4*)(a.part + min(j + u, a.splits - 1) * all + at);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (j + u < a.splits) s += t[u];
  }
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (a.bias) s[j] += (float)b[j];
    s[j] += r[j];
    o[j] = (bf16_t)s[j];
  }
  *(f32x4*)(a.res_out + at) = s;
  *(bf16x4*)(a.C + at) = o;
}

// Whether asking for W ahead pays (us, without | with, weights out of any cache; from the last-level cache it takes 3 - 8 % more wherever it is done, with few rows up to a third).
// Long contractions: 1 152 x 4 352, 196 rows 19.4 | 17.5, 729: 20.3 | 17.7, 1 024: 32.4 | 24.8; 768 x 3 072, 256: 16.1 | 13.4; not with 100 rows, 20.3 | 24.0: one tile of rows reads a line of W
// once in any case.  Two rounds of 128 x 128 tiles (tile 1): 5 120 x 2 048, 1 024 rows 39.8 | 34.2, 3 072 x 1 024, 1 458: 22.1 | 20.7; 2 x 5 632 x 2 048, 512: 41.8 | 38.0, 300: 35.6 | 37.4.  Others
// level at best: 1 152 x 1 152, 729 rows 6.7 | 7.3, 768 x 768: 5.6 | 6.2, 3 456 x 1 152: 14.9 | 14.0, 5 120 x 2 048: 22.8 | 23.5; 2 x 5 632 x 2 048, 200: 22.4 | 24.6.  Split: 2 048 x 7 680, 17
// rows 12.4 | 15.9, 200: 20.9 | 22.4, 300: 27.6 | 26.2, 768: 46 | 41.
bool asks_ahead(int epilogue, int tile, int64_t M, int K) {
  if (epilogue == EPI_PART) return K >= 3072 && M >= 288;
  if (tile == 1) return K >= 1024 && M >= (epilogue == EPI_GLU ? 512 : 192);
  return K >= 3072 && M >= 192 && epilogue != EPI_GLU;
}

template <int WM, int WN, int NS, int EPI>
int go_epi(GemmArgs& a, hipStream_t st) {
  constexpr int TM = 32 * WM, TO = EPI == EPI_GLU ? 16 * WN : 32 * WN, LDS = NS * (TM + 32 * WN) * 128;
  static const hipError_t attr = hipFuncSetAttribute((const void*)gemm_small_kernel<WM, WN, NS, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (attr != hipSuccess) {
    tv_set_error("gemm_small: cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  a.tiles_m = (a.M + TM - 1) / TM;
  a.tiles_n = (a.N + TO - 1) / TO;
  a.group_m = a.tiles_m < 4 ? a.tiles_m : 4;
  gemm_small_kernel<WM, WN, NS, EPI><<<dim3((unsigned)(a.tiles_m * a.tiles_n * (EPI == EPI_PART ? a.splits : 1))), GS_THREADS, LDS, st>>>(a);
  TV_LAUNCH_CHECK();
}
template <int WM, int WN, int NS>
int go(GemmArgs& a, int epilogue, hipStream_t st) {
  switch (epilogue) {
    case EPI_BIAS: return go_epi<WM, WN, NS, EPI_BIAS>(a, st);
    case EPI_BIAS_GELU: return go_epi<WM, WN, NS, EPI_BIAS_GELU>(a, st);
    case EPI_ACCUM: return go_epi<WM, WN, NS, EPI_ACCUM>(a, st);
    default: return go_epi<WM, WN, NS, EPI_GLU>(a, st);
  }
}

}  // namespace
}  // namespace tvgemm

extern "C" int tv_gemm_small_fwd(const void* A, const void* W, const void* bias, void* C, int64_t M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                                 int epilogue, int bias_dtype, int tile, void* stream) {
  using namespace tvgemm;
  TV_CHECK_ARG(A && W && C, "gemm_small: null pointer");
  TV_CHECK_ARG(M > 0 && N > 0 && K > 0 && tile >= 0 && tile <= 3, "gemm_small: bad sizes (M %lld N %d K %d, tile %d)", (long long)M, N, K, tile);
  TV_CHECK_ARG(epilogue == EPI_BIAS || epilogue == EPI_BIAS_GELU || epilogue == EPI_ACCUM || epilogue == EPI_GLU, "gemm_small: epilogue %d", epilogue);
  TV_CHECK_ARG(bias ? bias_dtype == TV_BF16 || (bias_dtype == TV_F32 && epilogue != EPI_GLU) : epilogue != EPI_GLU, "gemm_small: bias dtype %d", bias_dtype);
  if (K % BK || N % 8 || lda % 8 || ldw % 8 || ldc % 8 || lda < 0 || ldw < 0 || ldc < 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & 15) ||
      ((uintptr_t)bias & 15))
    TV_UNSUPPORTED("gemm_small: K must be a multiple of %d, N of 8, rows 16-byte aligned (K %d N %d lda %lld ldw %lld ldc %lld)", BK, K, N, (long long)lda,
                   (long long)ldw, (long long)ldc);
  if (M > (1ll << 24) || 128 * lda * 2 >= (1ll << 31) || ((epilogue == EPI_GLU ? (int64_t)N : 0) + 128) * ldw * 2 >= (1ll << 31) ||
      ((M + 63) / 64) * ((N + 31) / 32) >= (1ll << 31))
    TV_UNSUPPORTED("gemm_small: sizes beyond the 32-bit offsets of the copies");
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.bias = bias; a.C = (bf16_t*)C;
  a.M = (int)M; a.N = N; a.K = K; a.lda = lda; a.ldw = ldw; a.ldc = ldc;
  a.bias_f32 = bias_dtype == TV_F32;
  hipStream_t st = (hipStream_t)stream;
  // A tile whose work-groups are more than one round gives way to the next larger one if that fits a round (us: 1 152 x 4 352, 1 024 rows, 288 of 64 x 64 27.5, 144 of
  // 64 x 128 23.2; 3 456 x 1 152, 729 rows, 324 of 64 x 128 16.4, 162 of 128 x 128 12.1)
  const int64_t cus = tv_cu_count(), outs = epilogue == EPI_GLU ? 2ll * N : N;
  auto over = [&](int tm, int tn) { return ((M + tm - 1) / tm) * ((outs + tn - 1) / tn); };
  if (tile == 3 && over(64, 64) > cus && over(64, 128) <= cus) tile = 2;
  if (tile == 2 && over(64, 128) > cus && over(128, 128) <= cus) tile = 0;
  a.ahead = asks_ahead(epilogue, tile, M, K);
  switch (tile) {
    case 0: return go<4, 4, 4>(a, epilogue, st);
    case 1: return go<4, 4, 2>(a, epilogue, st);
    case 2: return go<2, 4, 4>(a, epilogue, st);
    default: return go<2, 2, 4>(a, epilogue, st);
  }
}

extern "C" size_t tv_gemm_small_add_workspace_bytes(int64_t M, int N, int splits) {
  return M > 0 && N > 0 && splits > 0 ? (size_t)splits * M * N * sizeof(float) : 0;
}

// Long contractions into few outputs, a few hundred rows: the contraction of each tile is split over work-groups, a second launch adds the splits, the bias and the residual stream.
extern "C" int tv_gemm_small_add_fwd(const void* A, const void* W, const void* bias, const float* residual, float* residual_out, void* C, int64_t M, int N, int K,
                                     int64_t lda, int64_t ldw, int tile, int splits, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace tvgemm;
  TV_CHECK_ARG(A && W && C && residual && residual_out, "gemm_small_add: null pointer");
  TV_CHECK_ARG(M > 0 && N > 0 && K > 0 && (tile == 0 || tile == 2 || tile == 3) && splits >= 1 && splits <= 64, "gemm_small_add: bad sizes (M %lld N %d K %d, tile %d, %d splits)",
               (long long)M, N, K, tile, splits);
  if (K % BK || K / BK < splits || N % 8 || lda % 8 || ldw % 8 || lda < 0 || ldw < 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || ((uintptr_t)C & 7) || ((uintptr_t)bias & 7) ||
      ((uintptr_t)residual & 15) || ((uintptr_t)residual_out & 15))
    TV_UNSUPPORTED("gemm_small_add: K must be a multiple of %d and of a step a split at least, N of 8, rows 16-byte aligned (K %d N %d lda %lld ldw %lld)", BK, K, N, (long long)lda,
                   (long long)ldw);
  if (M > (1ll << 24) || 128 * lda * 2 >= (1ll << 31) || 128 * ldw * 2 >= (1ll << 31) || ((M + 63) / 64) * ((N + 63) / 64) * splits >= (1ll << 31) || M * N / 4 >= (1ll << 31))
    TV_UNSUPPORTED("gemm_small_add: sizes beyond the 32-bit offsets of the copies");
  const size_t need = tv_gemm_small_add_workspace_bytes(M, N, splits);
  TV_CHECK_ARG(workspace && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0, "gemm_small_add: workspace of %zu bytes needed", need);
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.bias = bias; a.C = (bf16_t*)C;
  a.M = (int)M; a.N = N; a.K = K; a.lda = lda; a.ldw = ldw;
  a.part = (float*)workspace; a.splits = splits; a.res = residual; a.res_out = residual_out;
  a.ahead = asks_ahead(EPI_PART, tile, M, K);
  hipStream_t st = (hipStream_t)stream;
  const int rc = tile == 0 ? go_epi<4, 4, 4, EPI_PART>(a, st) : tile == 2 ? go_epi<2, 4, 4, EPI_PART>(a, st) : go_epi<2, 2, 4, EPI_PART>(a, st);
  if (rc != TV_OK) return rc;
  gemm_small_sum_kernel<<<dim3((unsigned)((M * N / 4 + 255) / 256)), 256, 0, st>>>(a);
  TV_LAUNCH_CHECK();
}
