// Products of a short prompt's rows with a weight matrix, y[m][n] = sum_k x[m][k] W[n][k], m <= 256: each weight byte is read once, for all
// rows, so that W from HBM is the floor (N K 2 bytes); at 256 rows the products are as long (1.3 PFLOP/s).
//
//   * A work-group owns 64, 96 or 128 rows of W and all rows of x; narrow outputs split K over work-groups as well, partial sums in fp32 to
//     a workspace and a second launch that adds them in order (the library runs 4 480 outputs on 35 - 70 of 256 compute units).
//   * Both operands arrive by LDS-DMA, a stage of 64 columns at a time.  Waves 0 - 3 copy x, waves 4 - 7 copy W: vmcnt counts in order, so a
//     wave that copied both would wait for W's latency with x.
//   * One barrier a stage, in the middle of its products: the fragments of a 16-column step are read while the step before is multiplied
//     (v_mfma_f32_32x32x16_bf16, W on the A side: a lane's registers are consecutive outputs of one row of x).
//   * The waves along K meet over the rings, in an order that stores whole rows of y.
//   * W past the caches (non-temporal), but for split matrices of up to 144 MB with 96 rows or more: work-groups that do not run in step ask for pieces of a row there, and plain loads are
//     better (nt_loads; us, best tiling each, non-temporal | plain, 203 rows: 4 480 x 5 120 29.1 | 27.9, 7 168 x 4 480 34.3 | 32.2, 4 480 x 10 240 39.0 | 37.9, 4 096 x 4 096, 160: 21.6 | 19.3; 65
//     rows and 4 480 x 15 680 level).  They are not beyond that or with rows that start 16 KiB apart (256 rows: 8 192 x 28 672 124 | 144, 16 384 x 16 384 145 | 181; 203 of 8 192 x 8 192
//     47.6 | 49.9), nor unsplit (22 656 x 4 480, 128 and 203 rows, 52.1 59.7 | 53.8 61.2; 64 rows 41.4 | 44.1).
// What bounds it: up to 64 rows the stream of W.  With 256 rows a stage of 128 rows of W takes 1.1 us, .8 of them where all copies hit the same lines, .57 without copies, .74 without
// fragment reads (copies dealt out between the products instead of in one burst change nothing); splits cost their sums' way through memory.
// fp32 accumulation, one rounding of y.
// Measured (weights not in any cache; library -> here): 4 480 x 15 680, 33 | 128 | 203 | 256 rows 65 | 89 | 131 | 148 -> 31 | 42 | 47 | 51 us; 4 480 x 10 240
// 52 | 57 | 83 | 92 -> 24 | 32 | 37 | 40; 15 680 x 4 480 with 33 | 64 | 96 rows 40 | 42 | 37 -> 28 | 32 | 35; 22 656 x 4 480, 128 | 256 55 | 73 -> 53 | 64.
#include "gemm_skinny.hpp"

namespace {
using namespace ssdk;

typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) const bf16x8 lds_bf16x8;
constexpr int GM_KC = 64;                          // columns of a stage
constexpr int GM_WAVES = 8;

// One of the up to three matrices that the rows of x meet in one launch: its tiles end in front of tile `end` of all
struct GmMat {
  const bf16_t* W;
  bf16_t* y;
  int N, end;
  int64_t ldw, ys;
};
struct GmArgs {
  const bf16_t *x, *bias;                          // (a bias: one matrix)
  GmMat m0, m1, m2;                                // (not an array: an index that is no constant would put the arguments into memory)
  float* part;                                     // split K: [split][M][all tiles' columns]
  int M, K, tiles, splits, per_xcd, relu2, nt;     // nt: W is read past the caches
  int64_t xs;
};
// the matrix of a tile, and the tile's place in it
__device__ __forceinline__ GmMat mat_of(const GmArgs& a, int& tile) {
  if (tile < a.m0.end) return a.m0;
  if (tile < a.m1.end) {
    tile -= a.m0.end;
    return a.m1;
  }
  tile -= a.m1.end;
  return a.m2;
}

// four consecutive outputs n.. of row m: bias, one rounding, squared ReLU of what was rounded
__device__ __forceinline__ void put(const GmArgs& a, const GmMat& w, int m, int n, f32x4 s) {
  if (a.bias) {
    const bf16x4 b = *(const bf16x4*)(a.bias + n);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] += (float)b[j];
  }
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    o[j] = (bf16_t)s[j];
    if (a.relu2) {
      const float r = fmaxf((float)o[j], 0.f);
      o[j] = (bf16_t)(r * r);
    }
  }
  *(bf16x4*)(w.y + (int64_t)m * w.ys + n) = o;
}

template <int J, bool NT>
__device__ __forceinline__ void glds_many(const void* src, const unsigned (&v)[J], unsigned dst) {
  if constexpr (J <= 4) glds_rows<J, NT>(src, v, dst);
  else {
    unsigned lo[4], hi[J - 4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = v[i];
#pragma unroll
    for (int i = 4; i < J; ++i) hi[i - 4] = v[i];
    glds_rows<4, NT>(src, lo, dst);
    glds_many<J - 4, NT>(src, hi, dst + 4096);
  }
}

// NI: 32-row tiles of W a work-group; waves: WM along the rows of x, MI tiles of 32 each, x WK along a stage's four 16-column steps;
// NSX, NSW: ring stages of x and of W
template <int NI, int MI, int WM, int WK, int NSX, int NSW>
__global__ __launch_bounds__(GM_WAVES * 64) void gemm_mid_kernel(GmArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char gm_smem[];
  static_assert(WM * WK == GM_WAVES && (WK == 2 || WK == 4), "waves");
  constexpr int XT = MI * WM, KS = 4 / WK;
  constexpr int XST = XT * 4096, WST = NI * 4096;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wk = wave / WM;
  const int r = lane & 31, hh = lane >> 5;
  // units (split, tile of N), tiles fastest: an XCD (id % 8) has a run of them, so that its work-groups share x's columns
  const int unit = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (unit >= a.tiles * a.splits) return;
  const int split = unit / a.tiles, tile = unit - split * a.tiles;
  int in_mat = tile;
  const GmMat mat = mat_of(a, in_mat);
  const int n0 = in_mat * (32 * NI);
  const int nst = a.K / GM_KC;
  const int s0 = (int)((int64_t)nst * split / a.splits), ns = (int)((int64_t)nst * (split + 1) / a.splits) - s0;

  // ---- copies: piece p (1 KiB), lane l -> LDS row 8 p + l / 8, 16-byte chunk l % 8, which holds source chunk (l % 8) ^ ((row >> 1) & 7)
  const bool xside = wave < 4;
  const unsigned ringx = lds_addr_of(gm_smem), ringw = ringx + (unsigned)(NSX * XST);
  unsigned vw[NI], vx[XT];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = 8 * ((wave & 3) * NI + i) + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    vw[i] = (unsigned)(((int64_t)min(row, mat.N - 1 - n0) * mat.ldw + ch * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < XT; ++i) {
    const int row = 8 * ((wave & 3) * XT + i) + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    vx[i] = (unsigned)(((int64_t)min(row, a.M - 1) * a.xs + ch * 8) * 2);
  }
  const bf16_t* Wb = mat.W + (int64_t)n0 * mat.ldw + (int64_t)s0 * GM_KC;
  const bf16_t* xb = a.x + (int64_t)s0 * GM_KC;
  f32x16_t acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[mi][ni][j] = 0.f;
  const bool busy = wm * MI * 32 < a.M;            // (rows past M: no products)
  unsigned fr[KS];                                 // fragment reads: row r of a 32-row tile, 16-byte chunk 2 ks + hh
#pragma unroll
  for (int k = 0; k < KS; ++k) fr[k] = (unsigned)(r * 128 + (((2 * (wk * KS + k) + hh) ^ ((r >> 1) & 7)) << 4));
  bf16x8 fx[2][MI], fw[2][NI];                     // two sets: the fragments of a step are read while the step before is multiplied
  auto read = [&](bf16x8 (&x)[MI], bf16x8 (&w)[NI], int k, int rx, int rw) __attribute__((always_inline)) {
    const unsigned px = ringx + (unsigned)(rx * XST) + fr[k] + (unsigned)(wm * MI * 4096), pw = ringw + (unsigned)(rw * WST) + fr[k];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) x[mi] = *(lds_bf16x8*)(size_t)(px + (unsigned)(mi * 4096));
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) w[ni] = *(lds_bf16x8*)(size_t)(pw + (unsigned)(ni * 4096));
  };
  auto multiply = [&](const bf16x8 (&x)[MI], const bf16x8 (&w)[NI]) __attribute__((always_inline)) {
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ni], x[mi], acc[mi][ni], 0, 0, 0);
  };
  // The loop of a wave that copies x (SIDE 0) or W (SIDE 1: past the caches, 2): J copies a stage into NS slots.  At a step's meeting stage i + 1 is in LDS for
  // all waves and every wave has read stage i, whose slot is filled again behind it.
  auto run = [&](auto side) __attribute__((always_inline)) {
    constexpr int SIDE = decltype(side)::value;
    constexpr bool XS = SIDE == 0;
    constexpr int NS = XS ? NSX : NSW, J = XS ? XT : NI, ST = XS ? XST : WST;
    const unsigned base = __builtin_amdgcn_readfirstlane((XS ? ringx : ringw) + 1024u * J * (wave & 3));
    auto issue = [&](int i, int slot) __attribute__((always_inline)) {
      const unsigned dst = __builtin_amdgcn_readfirstlane(base + (unsigned)(slot * ST));
      if constexpr (XS) glds_many<XT, false>(uniform_ptr(xb + (int64_t)i * GM_KC), vx, dst);
      else glds_many<NI, SIDE == 1>(uniform_ptr(Wb + (int64_t)i * GM_KC), vw, dst);
    };
    auto meet_counted = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(J * (NS - 2)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    auto meet_all = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    auto next = [](int v, int n) __attribute__((always_inline)) { return v == n - 1 ? 0 : v + 1; };
    for (int j = 0; j < NS - 1 && j < ns; ++j) issue(j, j);
    if (ns >= NS - 1) meet_counted();
    else meet_all();
    if (ns > NS - 1) issue(NS - 1, NS - 1);
    int i = 0, rx = 0, rw = 0, sl = 0;             // stage being multiplied; slots of the stage being read; slot of stage i in this wave's ring
    if (!busy) {
      for (; i + NS < ns; ++i) {
        meet_counted();
        issue(i + NS, sl);
        sl = next(sl, NS);
      }
      for (; i + 1 < ns; ++i) meet_all();
      return;
    }
    read(fx[0], fw[0], 0, 0, 0);
    if constexpr (KS == 2) {
      for (; i + NS < ns; ++i) {
        read(fx[1], fw[1], 1, rx, rw);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fx[0], fw[0]);
        meet_counted();
        issue(i + NS, sl);
        sl = next(sl, NS); rx = next(rx, NSX); rw = next(rw, NSW);
        read(fx[0], fw[0], 0, rx, rw);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fx[1], fw[1]);
      }
      for (; i + 1 < ns; ++i) {
        read(fx[1], fw[1], 1, rx, rw);
        multiply(fx[0], fw[0]);
        meet_all();
        rx = next(rx, NSX); rw = next(rw, NSW);
        read(fx[0], fw[0], 0, rx, rw);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fx[1], fw[1]);
      }
      read(fx[1], fw[1], 1, rx, rw);
      multiply(fx[0], fw[0]);
      multiply(fx[1], fw[1]);
    } else {
      for (; i + 1 + NS < ns; i += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          meet_counted();
          issue(i + u + NS, sl);
          sl = next(sl, NS); rx = next(rx, NSX); rw = next(rw, NSW);
          read(fx[1 - u], fw[1 - u], 0, rx, rw);
          __builtin_amdgcn_sched_barrier(0);
          multiply(fx[u], fw[u]);
        }
      }
      for (; i + 1 < ns; ++i) {
        if (i + NS < ns) {
          meet_counted();
          issue(i + NS, sl);
          sl = next(sl, NS);
        } else {
          meet_all();
        }
        rx = next(rx, NSX); rw = next(rw, NSW);
        read(fx[1], fw[1], 0, rx, rw);
        multiply(fx[0], fw[0]);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) fx[0][mi] = fx[1][mi];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) fw[0][ni] = fw[1][ni];
      }
      multiply(fx[0], fw[0]);
    }
  };
  if (xside) run(std::integral_constant<int, 0>{});
  else if (XT == 2 || a.nt) run(std::integral_constant<int, 1>{});
  else if constexpr (XT > 2) run(std::integral_constant<int, 2>{});
  // ---- the waves along K meet over the rings, MI rounds: [wave][n-tile][register quad][hh][r rotated] f32x4, summed in the order of rows of y
  f32x4* meet = (f32x4*)gm_smem;
  constexpr int NC = 8 * NI;                       // chunks of four outputs a row
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    __syncthreads();
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        meet[((wave * NI + ni) * 8 + 2 * g + hh) * 32 + ((r + 2 * g + hh + 8 * ni) & 31)] =
            f32x4{acc[mi][ni][4 * g], acc[mi][ni][4 * g + 1], acc[mi][ni][4 * g + 2], acc[mi][ni][4 * g + 3]};
    __syncthreads();
#pragma unroll
    for (int e0 = 0; e0 < WM * 32 * NC; e0 += GM_WAVES * 64) {
      const int e = e0 + tid, c = e % NC, row = e / NC, w = row >> 5, rr = row & 31;
      const int m = 32 * (w * MI + mi) + rr, n = n0 + 4 * c;
      f32x4 s = meet[(w * NC + c) * 32 + ((rr + c) & 31)];
#pragma unroll
      for (int k = 1; k < WK; ++k) s += meet[((k * WM + w) * NC + c) * 32 + ((rr + c) & 31)];
      if (m >= a.M) continue;
      if (a.part) *(f32x4*)(a.part + ((int64_t)split * a.M + m) * (a.tiles * 32 * NI) + tile * (32 * NI) + 4 * c) = s;
      else if (n < mat.N) put(a, mat, m, n, s);
    }
  }
}

// sum over the splits, in their order
__global__ __launch_bounds__(256) void gemm_mid_sum_kernel(GmArgs a, int width) {
  const int col = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4, m = blockIdx.y, np = a.tiles * width;
  if (col >= np) return;
  const bool first = col < a.m0.end * width, second = col < a.m1.end * width;
  const GmMat mat = first ? a.m0 : second ? a.m1 : a.m2;
  const int n = col - (first ? 0 : (second ? a.m0.end : a.m1.end) * width);
  if (n >= mat.N) return;
  const float* p = a.part + (int64_t)m * np + col;
  const int64_t step = (int64_t)a.M * np;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < a.splits; c += 4) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const f32x4*)(p + (int64_t)min(c + u, a.splits - 1) * step);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (c + u < a.splits) s += v[u];
  }
  put(a, mat, m, n, s);
}

template <int NI, int MI, int WM, int WK, int NSX, int NSW>
int launch_one(const GmArgs& a, hipStream_t st) {
  constexpr int RING = (NSX * MI * WM + NSW * NI) * 4096, MEET = GM_WAVES * NI * 4096;
  constexpr int LDS = RING > MEET ? RING : MEET;
  static_assert(LDS <= 160 * 1024, "ring");
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)gemm_mid_kernel<NI, MI, WM, WK, NSX, NSW>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (attr != hipSuccess) {
    tv_set_error("gemm_mid: cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  gemm_mid_kernel<NI, MI, WM, WK, NSX, NSW><<<dim3((unsigned)(8 * a.per_xcd)), GM_WAVES * 64, LDS, st>>>(a);
  if (a.part) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      tv_set_error("gemm_mid: %s", hipGetErrorString(e));
      return TV_ERR_LAUNCH;
    }
    gemm_mid_sum_kernel<<<dim3((unsigned)((a.tiles * 32 * NI + 1023) / 1024), (unsigned)a.M), 256, 0, st>>>(a, 32 * NI);
  }
  TV_LAUNCH_CHECK();
}

struct GmPlan {
  int ni, splits, xt;
};
// The tile width and split of K with the smallest estimate, us: a stage is a part for the rows of x and one for the 32-row tiles of W, which grows with the work-groups that stream W at once;
// each round of work-groups has its fill and epilogue, a launch its own; a split adds a second launch and 4 M N bytes written and read per split, and splits that start
// whole multiples of 4 KiB apart in a row meet in memory (4 480 x 10 240, 96 rows, five of 2 048 columns 33.6, seven 30.1; 16 384 x 8 192, 20 rows, two 64, unsplit 56).
// The numbers are a fit to all tilings of 47 sizes (N 1 024 to 32 768, K 4 096 to 28 672) with 20 to 256 rows, nothing in a cache, plain loads where nt_loads has them: over those 564 its choice is
// 1.0 % slower in the mean than the best one, 15 % at most, and 2.9 % faster than the estimate that took W and x through the compute unit's memory pipe at 45 bytes a ns, with its
// non-temporal loads (8.7 % slower at most, 4 096 x 8 192, 128 rows; a fit to 18 sizes with plain loads in all splits: up to 16 %, 8 192 x 28 672, 256 rows 124 | 144).
int tiles_of(int N, int ni) { return (N + 32 * ni - 1) / (32 * ni); }
GmPlan plan(int M, const int* N, int matrices, int K) {
  static constexpr double X[3] = {.047, .095, .36}, W[3] = {.048, .04, .056}, FILL[3] = {2., 3., .9};
  const int c = M <= 64 ? 0 : M <= 128 ? 1 : 2;
  GmPlan best{4, 1, 2 << c};
  const int cus = tv_cu_count(), nst = K / GM_KC;
  double least = 1e30, outs = 0;
  for (int i = 0; i < matrices; ++i) outs += N[i];
  for (int ni = 4; ni >= 2; --ni) {
    int64_t tiles = 0;
    for (int i = 0; i < matrices; ++i) tiles += tiles_of(N[i], ni);
    for (int s = 1; s <= 16 && (s == 1 || s * 8 <= nst); ++s) {
      const int64_t units = tiles * s, rounds = (units + cus - 1) / cus;
      const double stage = X[c] + ni * (W[c] + .097 * (units < cus ? units : cus) / cus);
      double t = rounds * (FILL[c] + (nst + s - 1) / s * stage) + 3.7;
      if (s > 1) t += 1.4 + s * (.09 + 1.26e-6 * outs * M);
      if (s > 1 && K / s * 2 % 4096 == 0) t *= 1.09;
      if (t < least) {
        least = t;
        best.ni = ni;
        best.splits = s;
      }
    }
  }
  return best;
}

template <int NI>
int launch_ni(const GmArgs& a, int xt, hipStream_t st) {
  if (xt == 2) return launch_one<NI, 1, 2, 4, 4, 32 / NI>(a, st);
  if (xt == 4) return launch_one<NI, 2, 2, 4, 3, 28 / NI>(a, st);
  return launch_one<NI, 2, 4, 2, 3, 16 / NI>(a, st);
}

bool nt_loads(int M, int64_t N, int K, int splits) { return splits == 1 || M < 96 || K % 8192 == 0 || N * K > 72000000; }

bool takes(const void* x, const void* W, int M, int N, int K, int64_t xs, int64_t ldw) {
  // (copies are 16 bytes a lane at 32-bit offsets from a work-group's first row; a stage is 64 columns; four outputs a store)
  return M >= 1 && M <= TV_GEMM_MID_MAX && N >= 4 && N % 4 == 0 && K >= GM_KC && K % GM_KC == 0 && xs % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x & 15) == 0 &&
         ((uintptr_t)W & 15) == 0 && xs >= 0 && ldw >= 0 && (int64_t)TV_GEMM_MID_MAX * xs * 2 < (1ll << 31) && 128 * ldw * 2 < (1ll << 31);
}

}  // namespace

extern "C" size_t tv_gemm_mid_multi_workspace_bytes(int M, const int* N, int matrices, int K) {
  if (M < 1 || M > TV_GEMM_MID_MAX || K < GM_KC || !N || matrices < 1 || matrices > 3) return 0;
  int64_t all = 0;
  for (int i = 0; i < matrices; ++i) {
    if (N[i] < 1) return 0;
    all += N[i];
  }
  if (all > 0x7fffffff) return 0;
  const GmPlan p = plan(M, N, matrices, K);
  int64_t tiles = 0;
  for (int i = 0; i < matrices; ++i) tiles += tiles_of(N[i], p.ni);
  return p.splits > 1 ? (size_t)p.splits * M * tiles * (128 * p.ni) : 0;
}

extern "C" size_t tv_gemm_mid_workspace_bytes(int M, int N, int K) { return tv_gemm_mid_multi_workspace_bytes(M, &N, 1, K); }

static int mid_go(const char* what, const void* x, const void* const* W, const void* bias, void* const* y, const int* N, int matrices, int M, int K,
                  int64_t x_stride, const int64_t* ldw, const int64_t* y_stride, int epilogue, void* workspace, size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(M >= 1 && M <= TV_GEMM_MID_MAX && K >= 1, "%s: M %d must be 1..%d, K %d positive", what, M, TV_GEMM_MID_MAX, K);
  TV_CHECK_ARG(epilogue == 0 || epilogue == TV_GEMM_ROWS_RELU2, "%s: epilogue %d", what, epilogue);
  int64_t all = 0;
  for (int i = 0; i < matrices; ++i) {
    TV_CHECK_ARG(x && W[i] && y[i], "%s: null pointer", what);
    TV_CHECK_ARG(N[i] >= 1, "%s: N %d must be positive", what, N[i]);
    if (!takes(x, W[i], M, N[i], K, x_stride, ldw[i]) || y_stride[i] % 4 || ((uintptr_t)y[i] & 7) || ((uintptr_t)bias & 7))
      TV_UNSUPPORTED("%s: K must be a multiple of %d, N and the row stride of y of 4, those of x and W of 8, x and W 16-byte, y and bias 8-byte aligned", what, GM_KC);
    all += N[i];
  }
  if (all > 0x7fffff00) TV_UNSUPPORTED("%s: %lld outputs", what, (long long)all);
  const GmPlan p = plan(M, N, matrices, K);
  const size_t need = tv_gemm_mid_multi_workspace_bytes(M, N, matrices, K);
  TV_CHECK_ARG(need == 0 || (workspace && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0), "%s: workspace of %zu bytes needed", what, need);
  GmArgs a{};
  a.x = (const bf16_t*)x; a.bias = (const bf16_t*)bias;
  a.M = M; a.K = K; a.xs = x_stride; a.relu2 = epilogue == TV_GEMM_ROWS_RELU2;
  GmMat* const to[3] = {&a.m0, &a.m1, &a.m2};
  for (int i = 0; i < 3; ++i) {
    if (i < matrices) {
      a.tiles += tiles_of(N[i], p.ni);
      *to[i] = GmMat{(const bf16_t*)W[i], (bf16_t*)y[i], N[i], 0, ldw[i], y_stride[i]};
    }
    to[i]->end = a.tiles;                                     // (a matrix that is not there has no tiles)
  }
  a.splits = p.splits;
  a.per_xcd = (a.tiles * a.splits + 7) / 8;
  a.part = p.splits > 1 ? (float*)workspace : nullptr;
  a.nt = nt_loads(M, all, K, p.splits);
  hipStream_t st = (hipStream_t)stream;
  switch (p.ni) {
    case 2: return launch_ni<2>(a, p.xt, st);
    case 3: return launch_ni<3>(a, p.xt, st);
    default: return launch_ni<4>(a, p.xt, st);
  }
}

extern "C" int tv_gemm_mid_fwd(const void* x, const void* W, const void* bias, void* y, int M, int N, int K, int64_t x_stride, int64_t ldw,
                               int64_t y_stride, int epilogue, void* workspace, size_t workspace_bytes, void* stream) {
  return mid_go("gemm_mid", x, &W, bias, &y, &N, 1, M, K, x_stride, &ldw, &y_stride, epilogue, workspace, workspace_bytes, stream);
}

// Up to three matrices in one launch.  An attention layer's q, k and v are 40 + 8 + 8 tiles of 256 compute units: 203 rows x (5 120, 1 024, 1 024) x 4 480, library, one by one |
// here 27 + 20 + 20 | 31 us.
extern "C" int tv_gemm_mid_multi_fwd(const void* x, const void* const* W, void* const* y, const int* N, int matrices, int M, int K, int64_t x_stride,
                                     const int64_t* ldw, const int64_t* y_stride, void* workspace, size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(W && y && N && ldw && y_stride && matrices >= 1 && matrices <= 3, "gemm_mid_multi: %d matrices, 1 to 3", matrices);
  return mid_go("gemm_mid_multi", x, W, nullptr, y, N, matrices, M, K, x_stride, ldw, y_stride, 0, workspace, workspace_bytes, stream);
}
