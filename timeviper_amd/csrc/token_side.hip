// What a token's own row of a second table adds behind a layer, y = P (gelu_tanh(G h) * e), in one launch: a narrow product, the gated row and the
// product back (G: 128 x D, P: D x 128).
//
// As three launches both products ran far below the chip's pace (128 outputs, or 128 columns of contraction: 17 us each for 6 011 rows, 2 048 wide) and a short
// prompt paid three calls.  A work-group takes 32 rows from h to y:
//   * G h: the eight waves split D in units of 32 columns, so that no operand is read twice; a unit (8 KB of G, 2 of h) arrives by LDS-DMA in a place of the wave's
//     own, is read into registers, and the next one is asked for in front of its products.  The partial sums meet in LDS.
//   * z = gelu_tanh(bf16(G h)) * e, rounded (what the separate launches write), stays in LDS.
//   * P z: a wave takes 32 outputs at a time (8 KB of P, two stages by LDS-DMA), whose rows are dealt to two tiles so that a lane holds eight neighbouring outputs:
//     16-byte stores.  With few rows several work-groups form the same z, each for a share of the outputs.
// G and P (1 MB) come from L2, read once a work-group: their latency and the way into the compute unit are what 32 rows take, so that the time hardly depends
// on the rows up to one round of work-groups (8 192 rows).  Loads straight into the matrix cores' layout, where neighbouring lanes are 16 different rows, took
// them in at 26 bytes a ns (a 16-byte access a lane): 46 us.
// Measured (2 048 wide; three launches -> here): 6 011 rows 40 -> 25 us on the device, 300 rows in one share 24.7, now 14.9; with the callers' host work, 40 to 1 000 rows 50 -> 23.
#include "gemm_skinny.hpp"

namespace {
using namespace ssdk;

constexpr int TS_ROWS = 32, TS_WAVES = 8, TS_DIM = 128;
constexpr int TILES = TS_DIM / 16, ITEMS = 2 * TILES * 64;             // pieces of z: four columns of a row
constexpr int UNIT = (TS_DIM + TS_ROWS) * 64;                          // bytes of 32 columns of G and h
constexpr int PAIR = 32 * TS_DIM * 2;                                  // bytes of 32 rows of P
constexpr int RING = TS_WAVES * ITEMS * 16;                            // (the partial sums: the largest of the three uses of the same bytes)
constexpr int ZROW = 2 * TS_DIM + 16;
constexpr int LDS = RING + TS_ROWS * ZROW;
static_assert(TS_WAVES * UNIT <= RING && TS_WAVES * 2 * PAIR <= RING && LDS <= 160 * 1024, "LDS");

struct SideArgs {
  const bf16_t *h, *G, *e, *P;
  const int64_t* ids;
  bf16_t* y;
  int64_t T, e_rows;
  int D;
  int64_t hs, gs, es, ps, ys;
};

__global__ __launch_bounds__(TS_WAVES * 64) void token_side_kernel(SideArgs a) {
  constexpr int KS = TS_DIM / 32, PER = ITEMS / (TS_WAVES * 64);
  extern __shared__ __attribute__((aligned(16))) unsigned char ts_smem[];
  typedef __attribute__((address_space(3))) const bf16x8 lds_bf16x8;
  f32x4* const part = (f32x4*)ts_smem;                                 // [wave][row half][tile][lane]
  unsigned char* const z = ts_smem + RING;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * TS_ROWS;
  const int left = (int)(a.T - row0 < TS_ROWS ? a.T - row0 : TS_ROWS);
  const unsigned lds0 = lds_addr_of(ts_smem);

  // ---- G h.  A copy moves 16 rows x 64 bytes: lane l to row l / 4, place l % 4, which holds 16-byte piece (l % 4) ^ (row / 4) (fragment reads of 16 rows
  // meet no bank twice); rows of h past the end repeat the last one
  unsigned vg[2][4], vh[2];
  {
    const int r = lane >> 2, c = (lane & 3) ^ ((r >> 2) & 3);
#pragma unroll
    for (int i = 0; i < 8; ++i) vg[i >> 2][i & 3] = (unsigned)(((16 * i + r) * (int)a.gs + 8 * c) * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) vh[i] = (unsigned)((min(16 * i + r, left - 1) * (int)a.hs + 8 * c) * 2);
  }
  const bf16_t* const hb = a.h + row0 * a.hs;
  const unsigned ring = lds0 + (unsigned)(wave * UNIT);
  auto copy = [&](int u) __attribute__((always_inline)) {
    glds_rows<4, false>(uniform_ptr(a.G + 32 * u), vg[0], ring);
    glds_rows<4, false>(uniform_ptr(a.G + 32 * u), vg[1], ring + 4096);
    glds_rows<2, false>(uniform_ptr(hb + 32 * u), vh, ring + 8192);
  };
  f32x4 acc[2][TILES];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < TILES; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int units = a.D / 32;
  if (wave < units) copy(wave);

  // this thread's pieces of the table's rows, on their way beside the first units
  bf16x4 ev[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int it = tid + i * TS_WAVES * 64, m = it / (TILES * 64), t = it / 64 % TILES, l = it & 63;
    const int64_t id = a.ids[row0 + min(16 * m + (l & 15), left - 1)];
    const bool ok = id >= 0 && id < a.e_rows;                          // (callers check ids on the host; a bad one counts as zeros)
    ev[i] = *(const bf16x4*)(a.e + (ok ? id : 0) * a.es + 16 * t + 4 * (l >> 4));
    if (!ok) ev[i] = bf16x4{};
  }

  const unsigned frag = ring + (unsigned)(n * 64 + ((kq ^ (n >> 2)) << 4));
  for (int u = wave; u < units; u += TS_WAVES) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bf16x8 hf[2], gf[TILES];
#pragma unroll
    for (int m = 0; m < 2; ++m) hf[m] = *(lds_bf16x8*)(size_t)(frag + (unsigned)(8192 + 1024 * m));
#pragma unroll
    for (int t = 0; t < TILES; ++t) gf[t] = *(lds_bf16x8*)(size_t)(frag + (unsigned)(1024 * t));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                 // (the next copies overwrite what has been read)
    __builtin_amdgcn_sched_barrier(0);
    if (u + TS_WAVES < units) copy(u + TS_WAVES);
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int m = 0; m < 2; ++m) acc[m][t] = mfma16(gf[t], hf[m], acc[m][t]);
  }
  __syncthreads();                                                     // every wave has left its unit
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int t = 0; t < TILES; ++t) part[((wave * 2 + m) * TILES + t) * 64 + lane] = acc[m][t];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int it = tid + i * TS_WAVES * 64, m = it / (TILES * 64), t = it / 64 % TILES, l = it & 63;
    f32x4 s = part[it];
#pragma unroll
    for (int w = 1; w < TS_WAVES; ++w) s += part[w * ITEMS + it];
    bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (bf16_t)(gelu_tanh_f((float)(bf16_t)s[r]) * (float)ev[i][r]);
    *(bf16x4*)(z + (16 * m + (l & 15)) * ZROW + 2 * (16 * t + 4 * (l >> 4))) = o;
  }
  __syncthreads();

  // ---- P z.  Row o of 32 rows of P belongs to row 4 (o / 8) + o % 4 of tile (o / 4) % 2.  A copy moves 4 rows x 256 bytes; a row's 16-byte pieces are exchanged by
  // its row in the tile
  bf16x8 zf[2][KS];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) zf[m][ks] = *(const bf16x8*)(z + (16 * m + n) * ZROW + 2 * (32 * ks + 8 * kq));
  unsigned vp[2][4];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int o = 4 * i + (lane >> 4), c = (lane & 15) ^ (4 * (o >> 3) + (o & 3));
    vp[i >> 2][i & 3] = (unsigned)((o * (int)a.ps + 8 * c) * 2);
  }
  const int npair = a.D / 32;
  const unsigned pring = lds0 + (unsigned)(wave * 2 * PAIR);
  auto copy_p = [&](int j, int S) __attribute__((always_inline)) {     // (past the end: the last rows again, so that the waits stay the same)
    const void* const src = uniform_ptr(a.P + (int64_t)(32 * min(j, npair - 1)) * a.ps);
    glds_rows<4, false>(src, vp[0], pring + (unsigned)(S * PAIR));
    glds_rows<4, false>(src, vp[1], pring + (unsigned)(S * PAIR + 4096));
  };
  const int first = wave + TS_WAVES * (int)blockIdx.y, step = TS_WAVES * (int)gridDim.y;
  copy_p(first, 0);
  copy_p(first + step, 1);
  const unsigned pfrag = (unsigned)((8 * (n >> 2) + (n & 3)) * 256);
  int S = 0;
  for (int j = first; j < npair; j += step, S ^= 1) {
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");                   // (the younger stage stays in flight; stores among it make the wait stricter)
    bf16x8 pf[2][KS];
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        pf[half][ks] = *(lds_bf16x8*)(size_t)(pring + (unsigned)(S * PAIR + 1024 * half) + pfrag + (unsigned)(((4 * ks + kq) ^ n) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    copy_p(j + 2 * step, S);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      f32x4 o[2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        o[half] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) o[half] = mfma16(pf[half][ks], zf[m][ks], o[half]);
      }
      bf16x8 v;
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = (bf16_t)o[r >> 2][r & 3];
      if (16 * m + n < left) *(bf16x8*)(a.y + (row0 + 16 * m + n) * a.ys + 32 * j + 8 * kq) = v;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                     // no copy may land in another work-group's LDS
}

}  // namespace

extern "C" int tv_token_side_fwd(const void* h, const int64_t* ids, const void* table, const void* gate, const void* proj, void* y, int64_t rows, int width,
                                 int dim, int64_t table_rows, int64_t h_stride, int64_t table_stride, int64_t gate_stride, int64_t proj_stride,
                                 int64_t y_stride, void* stream) {
  TV_CHECK_ARG(rows >= 0 && rows < (1ll << 31) && width > 0 && dim > 0 && table_rows > 0, "token_side: bad sizes");
  if (rows == 0) return TV_OK;
  TV_CHECK_ARG(h && ids && table && gate && proj && y, "token_side: null pointer");
  if (width % 32 || dim != TS_DIM || h_stride % 8 || gate_stride % 8 || proj_stride % 8 || y_stride % 8 || table_stride % 4 || ((uintptr_t)h & 15) ||
      ((uintptr_t)gate & 15) || ((uintptr_t)proj & 15) || ((uintptr_t)y & 15) || ((uintptr_t)table & 7))
    TV_UNSUPPORTED("token_side: width must be a multiple of 32, dim %d, rows 16-byte aligned (the table's 8-byte)", TS_DIM);
  if (h_stride < 0 || gate_stride < 0 || proj_stride < 0 || h_stride >= (1 << 22) || gate_stride >= (1 << 22) || proj_stride >= (1 << 22))
    TV_UNSUPPORTED("token_side: rows more than 2^22 elements apart");
  SideArgs a;
  a.h = (const bf16_t*)h; a.G = (const bf16_t*)gate; a.e = (const bf16_t*)table; a.P = (const bf16_t*)proj; a.ids = ids; a.y = (bf16_t*)y;
  a.T = rows; a.e_rows = table_rows; a.D = width;
  a.hs = h_stride; a.gs = gate_stride; a.es = table_stride; a.ps = proj_stride; a.ys = y_stride;
  static const hipError_t attr = hipFuncSetAttribute((const void*)token_side_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (attr != hipSuccess) {
    tv_set_error("token_side: cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  // Work-groups a block of rows, each with a share of the outputs, where that keeps within three quarters of the compute units (2 048 wide, us by shares 1 | 2 | 4 | 8: 300 rows
  // 24.7 19.3 16.2 14.9, 1 000, 8 of which are a work-group on every unit, 22.9 18.1 16.0 17.9, 1 500 22.7 18.7 18.5 31.9, 4 100 24.5 35.4): as many as shorten the longest share
  const int64_t blocks = (rows + TS_ROWS - 1) / TS_ROWS, turns = (width + 32 * TS_WAVES - 1) / (32 * TS_WAVES);
  int64_t shares = tv_cu_count() * 3 / 4 / blocks;
  shares = shares > 8 ? 8 : shares < 1 ? 1 : shares;
  const int64_t longest = (turns + shares - 1) / shares;
  shares = (turns + longest - 1) / longest;
  token_side_kernel<<<dim3((unsigned)blocks, (unsigned)shares), TS_WAVES * 64, LDS, (hipStream_t)stream>>>(a);
  TV_LAUNCH_CHECK();
}
