// A1 / T3 / ViT: fused softmax attention forward on CDNA4 MFMA tiles.
//
// Structure (wave64, v_mfma_f32_32x32x16): a workgroup of 8 waves owns 256 query
// rows of one (batch, q-head) (128 with half of the keys a wave where those are too few work-groups; 4 waves for 128 rows of many short ones); each wave keeps
// its 32 query rows as MFMA B fragments in registers for the whole kernel.  K/V tiles
// of 64 keys arrive by LDS-DMA into rings of four shared by the waves, a step of two tiles
// ahead of the math, one barrier a step.  A wave's loop is pipelined over its tiles: the
// next tile's scores are multiplied beside the present one's exponentials.  The score tile is computed
// TRANSPOSED, S^T = K . Q^T, so every lane owns one query column: the softmax
// row statistics are per-lane scalars (one cross-half shuffle per tile), and the
// P^T accumulator registers are, after a bf16 pack, directly the B operand of
// O^T += V^T . P^T — V^T fragments come from the row-major V tile through the
// gfx950 transposing LDS read (ds_read_b64_tr_b16).  No S x S matrix, no
// repeat_kv copy for GQA, exp2-domain online softmax in fp32.
//
// Reference semantics: _flash_attention_forward (modeling_nano.py:1198-1209,
// causal, no positional encoding, scale 1/sqrt(d)), SDPA (:1300-1307,
// cross_attention.py:310-317 non-causal), flash_attn_varlen_qkvpacked_func
// (flash_attention_class.py:59-66).
#include "ssd_common.hpp"
#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

constexpr int FA_QW = 32;                  // query rows per wave
constexpr int FA_KT = 3;                   // key sub-tiles of 32 per LDS tile of the streaming kernels and of rows that see one tile

typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Fragment reads take a 32-bit LDS byte offset: one base register per fragment family and iteration,
// everything compile-time (sub-tile, k-step, row half) in the instruction's offset field.  (With generic
// pointers hipcc spent a v_add per read: 112 of the ~330 VALU instructions of a ViT tile, in a loop
// that is VALU-bound at head_dim 72.)
typedef __attribute__((address_space(3))) unsigned char lds_u8;
__device__ __forceinline__ const lds_u8* lds_at(unsigned off) { return (const lds_u8*)(uintptr_t)off; }

using ssdk::u32x4;
using ssdk::gload16_async;
using ssdk::settle;

// f(integral_constant) for FROM .. TO - 1: indices into register arrays have to be constants
template <int FROM, int TO, typename F> __device__ __forceinline__ void static_for(F&& f) {
  if constexpr (FROM < TO) {
    f(std::integral_constant<int, FROM>{});
    static_for<FROM + 1, TO>(f);
  }
}

template <typename T> struct Frag;
template <> struct Frag<bf16_t> {
  typedef bf16x8 v8; typedef bf16x4 v4; typedef bf16_t v2 __attribute__((ext_vector_type(2)));
  static constexpr bool is_bf16 = true;
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ v4 tr_read(const lds_u8* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
  }
  static __device__ __forceinline__ v8 row_read(const lds_u8* p) {
    return *(const __attribute__((address_space(3))) v8*)p;
  }
};
template <> struct Frag<f16_t> {
  typedef f16x8 v8; typedef f16x4 v4; typedef f16_t v2 __attribute__((ext_vector_type(2)));
  static constexpr bool is_bf16 = false;
  static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ v4 tr_read(const lds_u8* p) {
    const s16x4 raw = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
    return __builtin_bit_cast(f16x4, raw);
  }
  static __device__ __forceinline__ v8 row_read(const lds_u8* p) {
    return *(const __attribute__((address_space(3))) v8*)p;
  }
};

struct AttnArgs {
  const void *q, *k, *v;
  void* o;
  float* lse;
  int Lq, Lk, Hq, Hkv, D;
  int64_t qsb, qsl, qsh, ksb, ksl, ksh, vsb, vsl, vsh, osb, osl, osh;
  float scale_log2;  // softmax_scale * log2(e)
  int causal;
  int nqb, nb;       // nqb > 0: many short sequences, nqb query blocks per (batch, head); 0: blocks dealt out by block_of; nb batches
  int ppx;           // streaming kernel: (batch, head) pairs per XCD
  int o16;           // streaming kernel: o rows are 16-byte aligned (wide epilogue stores)
  int Dv;            // value head dim (D unless the caller says otherwise)
  const float* sink; // per q-head logit without key or value that joins the denominator, or NULL (flash_fwd_kernel, causal)
  int window, keep;  // flash_fwd_kernel with WIN: position p sees keys (p - window, p] and the first `keep`
  const void* gate;  // WIN: o is multiplied by sigmoid(gate), element by element, or NULL
  int64_t gsl, gsh;
  int notrim;        // streaming kernel (dev, TV_FA_TRIM=0): the last key tile runs all its sub-tiles
};

// Sequences of a packed step (WIN): rows [row, row + len_q) of q, o and gate against the first len_k rows of batch entry `slot`
constexpr int FA_SEQS = 32;
struct AttnSeqs {
  int row[FA_SEQS], len_q[FA_SEQS], len_k[FA_SEQS], slot[FA_SEQS];
};
struct NoSeqs {};

// Work-group `id` of a grid of query blocks x (batch, head) pairs, the pairs fastest: block `t` of `pair`.  A causal block's cost
// grows with its position, so the blocks of all heads are dealt out by falling cost (a grid that finishes one head after
// the other ends with the last heads' heaviest blocks running alone: 40 heads x 5 003 tokens 402 us, dealt out 309; 10 007 tokens: 1 475, 1 215).
// An XCD (id % 8) gets a contiguous range of the pairs in every round, about the same one: heads that share K / V share an L2.
// SCALAR: the quotient, and with it all addresses, in scalar registers (a division leaves it in a vector register): 64 rows against 4 064 keys, 16
// heads on 4 x 128, windowed: 58.4 us, so 57.2; the plain kernels have no scalar registers to spare (16 x 16 000: 461, so 472).
template <bool SCALAR>
__device__ __forceinline__ void block_of(int id, int pairs, int& t, int& pair) {
  t = SCALAR ? __builtin_amdgcn_readfirstlane(id / pairs) : id / pairs;
  const int p = id - t * pairs, q = pairs >> 3, rem = pairs & 7;
  const int x0 = (id - p) & 7, x = id & 7;             // XCD of the round's first work-group, and of this one
  // an XCD gets q pairs of a round, the `rem` XCDs from x0 on (modulo 8) one more: those in front of XCD x
  const int more = x0 + rem <= 8 ? min(max(x - x0, 0), rem) : min(x, x0 + rem - 8) + max(x - x0, 0);
  pair = x * q + more + (p >> 3);
}

// ssdk::glds16 for the lanes of `live` only (a wave-uniform mask): the other lanes' 16 LDS bytes keep what they hold.  (Five wait states in front of the load, as there.)
__device__ __forceinline__ void glds16_lanes(const void* sbase, unsigned voff, unsigned lds_dst, unsigned long long live) {
  unsigned keep;
  unsigned long long ex;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_mov_b64 %1, exec\n\ts_mov_b64 exec, %5\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, %1\n\ts_mov_b32 m0, %0"
               : "=&s"(keep), "=&s"(ex) : "v"(voff), "s"(sbase), "s"(lds_dst), "s"(live) : "memory");
}

// KS = ceil(D/16) k-steps of QK^T, DT = ceil(D/32) d-tiles of PV, NW waves per workgroup.
// K/V tiles of 32*KT keys go global -> LDS by LDS-DMA (global_load_lds_dwordx4, 16 bytes per
// lane, no VGPR round trip: staging through registers cost a third of the kernel) into
// rings of four tiles, a step of two tiles ahead of the math, one copy instruction every few MFMAs (a step's 64 in a row hold up every wave: 5 003 tokens, 40 heads: 330 us,
// spread 304).  One barrier a step: with one per tile of 64 keys and rings of three 345 us.
// What bounds it: long grids the chip's power (16 384 tokens: the matrix pipe is busy .62 of the time at 1.83 GHz, where one phase behind the other, all waves between
// the same barriers, it was .48 at 2.09), short ones the chain of steps.  us, before and with this loop, causal, 40 heads on 8 x 128: 1 400 tokens 53 | 45, 5 003 308 | 280,
// 16 384 2 725 | 2 455; 16 heads of 64, 4 096: 81 | 61; of 80: 94 | 70; windows of 256 - 8 192 in 2 - 16 prompts: 1.07 - 1.5 times.
// LDS rows are 256 bytes (128 elements); the 16-byte chunks of a row are
// XOR-swizzled on the DMA source address so that the row reads of K (ds_read_b128, chunk ^
// row%16) and the transposing reads of V (ds_read_b64_tr_b16, chunk ^ 4(row%4)) are bank
// conflict free.  Chunks past head_dim are never copied (the K ones QK^T reads are zeroed once).
// KG 2: the first four waves and the last four hold the same 128 query rows and take every second tile of 32 KT keys each, one of a step's two; the halves (maximum, sum, accumulators) meet in LDS at the end.  A short grid is a chain of steps that lasts as long as the longest row of keys: this
// halves it with the same two waves a SIMD (1 100 tokens, 40 heads: 35.2 -> 31.2 us).  Long grids lose by it: K and V go into LDS once per 128 rows.
// WIN: causal with a sliding window and kept first keys.  The work-group visits the tiles that hold kept keys, then jumps to the
// first tile of its first row's window: ring, copies and waits count the visited tiles.  All sequences of a packed step share the
// launch (a launch per prompt leaves most of the chip idle: six prompts, 6 011 tokens, 16 heads on 4 x 128, window 1 024: 265 us, in one launch 95).
// A step's copies stand between its MFMAs, copy c behind number (2 c + 1) n / (2 copies) of n: how many of them in front of number i
constexpr int copies_before(int i, int n, int copies) {
  int c = 0;
  while (c < copies && (2 * c + 1) * n / (2 * copies) < i) ++c;
  return c;
}
constexpr int fa_slots(int kt) { return kt == 2 ? 4 : 1; }                       // (KT 3: keys of one tile)
constexpr int fa_lds(int kt) { return 2 * fa_slots(kt) * 32 * kt * 256; }      // K and V rings, rows of 256 bytes
template <typename T, int KS, int DT, int NW, int KT, bool WIN = false, int KG = 1>
__global__ __launch_bounds__(NW * 64) void flash_fwd_kernel(AttnArgs a, typename std::conditional<WIN, AttnSeqs, NoSeqs>::type sq) {
  constexpr int FA_KB = 32 * KT;     // keys per tile
  constexpr int TPK = FA_KB / 4;     // 1 KiB DMA pieces (4 key rows) of K per tile
  typedef typename Frag<T>::v8 v8;
  typedef typename Frag<T>::v4 v4;
  typedef typename Frag<T>::v2 v2;
  constexpr int QB = NW / KG * FA_QW;     // query rows per workgroup
  constexpr int ROWB = 256;          // LDS bytes per key row
  constexpr int TILEB = FA_KB * ROWB;
  constexpr int SLOTS = fa_slots(KT);           // tiles of the rings
  static_assert(SLOTS == 1 || (SLOTS == 4 && TILEB == 16384), "a ring's halves are bit 15 of an LDS address");
  constexpr int TPS = KG == 1 ? 2 : 1;          // tiles of a step that one wave takes: a step is two tiles
  extern __shared__ __attribute__((aligned(16))) unsigned char fa_smem[];
  unsigned char* const sK = fa_smem;
  const unsigned sK_off = (unsigned)(uintptr_t)(lds_u8*)fa_smem, sV_off = sK_off + SLOTS * TILEB;      // (sK_off is 0: all LDS is dynamic)

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 31, hh = lane >> 5;
  // 1-D grid.  Few sequences: `block_of` (causal: the heaviest query blocks of all heads first).  Many short sequences (ViT
  // frames): ids walk the query blocks of ONE (batch, head) on one XCD (id % 8): the blocks that
  // share K / V then share an L2 instead of pulling the same keys into three of them
  int qblk, h, b, Lq = a.Lq, Lk = a.Lk;
  int64_t row0 = 0;                             // WIN: the sequence's first row of q, o and gate
  if constexpr (WIN) {
    int t;
    block_of<true>(blockIdx.x, a.Hq, t, h);
    int s = 0, nblk;
    for (;; ++s) {                              // (t is below the sum of the sequences' blocks: launcher)
      nblk = (sq.len_q[s] + QB - 1) / QB;
      if (t < nblk) break;
      t -= nblk;
    }
    qblk = nblk - 1 - t;
    Lq = sq.len_q[s];
    Lk = sq.len_k[s];
    row0 = sq.row[s];
    b = sq.slot[s];
  } else if (a.nqb > 0) {
    const int slot = blockIdx.x >> 3;
    // an XCD owns a contiguous range of (batch, head) pairs: neighbouring heads of a frame interleave
    // in memory (head_dim 72 = 144-byte rows inside 128-byte lines), so their shared lines hit one L2
    const int pair = (blockIdx.x & 7) * (int)(gridDim.x / (8 * a.nqb)) + slot / a.nqb;
    qblk = slot % a.nqb;
    h = pair % a.Hq;
    b = pair / a.Hq;
    if (b >= a.nb) return;                    // (batch, head) pairs are padded to a multiple of 8
  } else if constexpr (NW == 4) {               // short sequences: one block each, a grid of heads and batch entries
    qblk = 0;
    h = blockIdx.y;
    b = blockIdx.z;
  } else {
    const int pairs = a.nb * a.Hq;
    int pair;
    block_of<KG == 2>(blockIdx.x, pairs, qblk, pair);
    if (a.causal) qblk = (a.Lq + QB - 1) / QB - 1 - qblk;
    b = a.nb == 1 ? 0 : pair / a.Hq;           // (a division is 30 instructions of a short call)
    if (KG == 2) b = __builtin_amdgcn_readfirstlane(b);
    h = pair - b * a.Hq;
  }
  const int hk = WIN || KG == 2 ? __builtin_amdgcn_readfirstlane(h / (a.Hq / a.Hkv)) : h / (a.Hq / a.Hkv);
  const int grp = KG == 1 ? 0 : wave / (NW / KG);                        // which of a step's tiles this wave takes
  const int q0 = qblk * QB + (wave - grp * (NW / KG)) * FA_QW;      // first query row of this wave
  const int qrow = q0 + r;                      // this lane's query row
  const int D = a.D;
  const int shift = Lk - Lq;                // bottom-right causal alignment

  const T* qp = (const T*)a.q + (WIN ? row0 * a.qsl : (int64_t)b * a.qsb) + (int64_t)h * a.qsh;
  const T* kp = (const T*)a.k + (int64_t)b * a.ksb + (int64_t)hk * a.ksh;
  const T* vp = (const T*)a.v + (int64_t)b * a.vsb + (int64_t)hk * a.vsh;

  // K chunks between head_dim and the padded 16*KS columns are read by QK^T (against zero Q
  // columns) but never copied: zero them once so that stale LDS bits cannot be NaN/Inf.  (V
  // chunks past head_dim only feed output rows that are never stored.)
  if (D < 16 * KS) {
    const v8 z = {};
    const int c0 = D / 8, nc = 2 * KS - c0;
    for (int i = tid; i < SLOTS * FA_KB * nc; i += NW * 64) {
      const int row = i / nc, c = c0 + i % nc;
      *reinterpret_cast<v8*>(sK + row * ROWB + ((c ^ (row & 15)) << 4)) = z;
    }
  }

  // Q^T fragments (B operand): lane (r,hh) holds Q[qrow][16ks + 8hh + j]; untracked loads, settled
  // behind the first counted wait below
  v8 qf[KS];
  u32x4 qraw[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 16 + hh * 8;
    qraw[ks] = gload16_async((qrow < Lq && d0 < D) ? qp + (int64_t)qrow * a.qsl + d0 : qp);
  }

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // key range this workgroup needs
  const int wg_q_last = min(qblk * QB + QB, Lq) - 1;
  int k_end = a.causal ? min(Lk, wg_q_last + shift + 1) : Lk;
  if (k_end < 0) k_end = 0;
  int ntiles = (k_end + FA_KB - 1) / FA_KB;
  int tkeep = 0, tskip = 0;                     // WIN: visited tile i is tile i, or i + tskip from tkeep on
  if constexpr (WIN) {
    tkeep = (min(a.keep, k_end) + FA_KB - 1) / FA_KB;
    tskip = max(max(0, qblk * QB + shift - a.window + 1) / FA_KB - tkeep, 0);
    ntiles -= tskip;
  }
  auto key_of_tile = [&](int kt) __attribute__((always_inline)) { return (WIN && kt >= tkeep ? kt + tskip : kt) * FA_KB; };

  constexpr bool FEW = KS > 6 && WIN;           // no registers left: lane constants of the loop are formed where they are used
  // ---- copies: a tile is TPK pieces of 4 key rows (lane l: row l / 16, LDS slot l % 16), piece wave + NW j of it this wave's; the rows of a wave's pieces are
  // 4 NW apart, a multiple of 16, so that one lane offset an operand serves all of them (the source pointer moves instead)
  constexpr int PPT = TPK / NW;                 // pieces of a tile this wave copies
  static_assert(TPK % NW == 0 && 4 * NW % 16 == 0, "pieces must divide over the waves");
  const int c_row = 4 * wave + (lane >> 4);
  const int ck = (lane & 15) ^ (c_row & 15), cv = (lane & 15) ^ (4 * (c_row & 3));      // source chunks
  const unsigned long long k_live = __builtin_amdgcn_ballot_w64(ck < a.D / 8), v_live = __builtin_amdgcn_ballot_w64(cv < a.Dv / 8);      // (chunks past the head dim: nothing to copy)
  const unsigned k_row = (unsigned)a.ksl * (unsigned)sizeof(T), v_row = (unsigned)a.vsl * (unsigned)sizeof(T);      // (below 2^24: launcher)
  auto copy_piece = [&](bool isK, int tile, int j) __attribute__((always_inline)) {      // (no branch: a tile that does not exist has no lanes)
    const int kbase = key_of_tile(tile);
    const void* src = ssdk::uniform_ptr(isK ? kp + (int64_t)kbase * a.ksl : vp + (int64_t)kbase * a.vsl);
    int cr = c_row, cc = isK ? ck : cv;
    if constexpr (FEW) {
      int l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
      asm volatile("" : "+v"(l));
      cr = 4 * wave + (l >> 4);
      cc = (l & 15) ^ (isK ? cr & 15 : 4 * (cr & 3));
    }
    const int row = min(cr + 4 * NW * j, Lk - kbase - 1);                                   // rows past the end repeat the last key (masked later)
    const unsigned off = __umul24((unsigned)row, isK ? k_row : v_row) + (unsigned)(cc * 16);
    glds16_lanes(src, off, __builtin_amdgcn_readfirstlane((isK ? sK_off : sV_off) + (unsigned)(tile % SLOTS * TILEB + (wave + NW * j) * 1024)), tile < ntiles ? isK ? k_live : v_live : 0ull);
  };
  auto copy_tile = [&](bool isK, int tile) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PPT; ++j) copy_piece(isK, tile, j);
  };
  // what the step that starts with this wave's tile kt copies: the next one's tiles, piece c of 4 PPT
  auto copy_ahead = [&](int kt, int c) __attribute__((always_inline)) {
    const int t = c / PPT, tile = kt * KG + (t & 1);
    copy_piece(t < 2, tile + (t < 2 ? KG + 2 : 2), c % PPT);
  };

  // fragment reads: LDS addresses in the ring's present half (bit 15; KG 2: in this wave's tile of it); tile and sub-tile are instruction offsets
  constexpr int NK = FEW ? 1 : KS, NV = FEW ? 1 : DT;
  unsigned k_rd[NK], v_rd[NV];
  constexpr unsigned HALF = SLOTS == 4 ? 2 * TILEB : 0;
  auto set_reads = [&](unsigned half) __attribute__((always_inline)) {
    const int kz = (hh ^ (r & 15)) << 4;      // K row fragment: row t*32 + r, chunk (2ks + hh) ^ (r % 16)
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) k_rd[ks] = sK_off + half + (unsigned)(grp * TILEB + r * ROWB + ((32 * ks) ^ kz));
    const int q4 = (lane & 15) >> 2, p4 = lane & 3, cc = 2 * ((lane >> 4) & 1) + (p4 >> 1);      // V^T fragment: row 16s + 4hh + q4 (+8), chunk (4dt + cc) ^ 4 q4
#pragma unroll
    for (int dt = 0; dt < NV; ++dt) v_rd[dt] = sV_off + half + (unsigned)(grp * TILEB + (4 * hh + q4) * ROWB + ((4 * (dt ^ q4) + cc) << 4) + (p4 & 1) * 8);
  };

  // ---- the steps this wave works in: of the visited tiles [0, n_seen) start below the last key its rows see; a window leaves out those between the kept keys and
  // its first row's window
  const int wave_q_last = q0 + FA_QW - 1;
  int n_seen = ntiles, keep_to = 0, win_from = 0;
  if (a.causal) {
    const int whole = wave_q_last + shift < 0 ? 0 : (wave_q_last + shift) / FA_KB + 1;       // tiles of the sequence that start at or below it
    n_seen = min(ntiles, WIN ? (whole <= tkeep ? whole : max(tkeep, whole - tskip)) : whole);
  }
  if (q0 >= Lq) n_seen = 0;
  if constexpr (WIN) {
    keep_to = min(tkeep, n_seen);
    win_from = max(keep_to, min(n_seen, max(0, q0 + shift - a.window + 1) / FA_KB - tskip));
  }
  // a wave's own count of tiles: with two waves a row every second one is its own
  auto own = [&](int tile) __attribute__((always_inline)) { return KG == 1 ? tile : (max(tile - grp, 0) + KG - 1) / KG; };
  const int nown = (ntiles + KG - 1) / KG;

  __syncthreads();                 // LDS zeroed before the first copy lands
  // K of the first tile (of both halves) has landed, and Q, older, behind the first wait; the rest of the first step may be in flight
  copy_tile(true, 0);
  if (KG == 2) copy_tile(true, 1);
  if constexpr (SLOTS > 1) { copy_tile(true, KG); copy_tile(true, KG + 1); }
  copy_tile(false, 0);
  if constexpr (SLOTS > 1) copy_tile(false, 1);
  if (SLOTS > 1 && ntiles > KG + 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * PPT) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (copies without lanes are not counted on)
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    settle(qraw[ks]);
    const v8 z = {};
    qf[ks] = (qrow < Lq && ks * 16 + hh * 8 < D) ? __builtin_bit_cast(v8, qraw[ks]) : z;
  }

  // ---- a step: the scores of the wave's next tile (Q.K^T, matrix pipe) beside the weights of the present one (exponentials, vector pipe), then its P.V beside the
  // next tile's maximum.  Every MFMA (32 cycles) gets its share of vector work in the source order, which the scheduling barriers pin: a wave keeps both pipes
  // busy by itself, and its partner on the SIMD fills what is left.  (Multiplying first and exponentiating behind it, all waves between the same two barriers:
  // 7 000 cycles a tile of 96 keys where the matrix pipe needs 3 072.)
  // The accumulators are rescaled whenever some row's maximum has moved: a maximum that follows only when it has grown by 2^8 saves nearly all of that (5 003 tokens,
  // 40 heads: 329 -> 305 us), but then a row's largest weight is no longer exactly 1 in bf16, and the error against 64 bits grows from .0019 to .0022.
  constexpr int NQK = KT * KS, NPV = 2 * KT * DT, NE = 16 * KT;
  constexpr int NE1 = NE * 5 / 8 / 2 * 2;       // weights formed beside Q.K^T, the rest beside P.V, each in front of the k-step that needs it
  constexpr int LEAD = 4;                       // ... of them ahead of the first MFMA, whose operands are still on their way from LDS
  constexpr int KAHEAD = FEW && KG == 2 ? 2 : 4;                     // K fragments read ahead
  float neg_m = 0.f;                            // - maximum, 0 while there is none
  typedef f32x16 Scores[KT];
  Scores s0, s1;
  auto tile_key = [&](int kt) __attribute__((always_inline)) { return key_of_tile(KG == 1 ? kt : kt * KG + grp); };
  auto mask = [&](int kt, Scores& S) __attribute__((always_inline)) {
    const int kbase = tile_key(kt);
    bool need = (kbase + FA_KB > Lk) || (a.causal && kbase + FA_KB - 1 > q0 + shift);
    if constexpr (WIN) need = need || (kbase <= wave_q_last + shift - a.window && kbase + FA_KB > a.keep);
    if (need) {
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = kbase + t * 32 + (i & 3) + 8 * (i >> 2) + 4 * hh;
          bool ok = key < Lk && (!a.causal || key <= qrow + shift);
          if constexpr (WIN) ok = ok && (key > qrow + shift - a.window || key < a.keep);
          S[t][i] = ok ? S[t][i] : -INFINITY;
        }
    }
  };
  auto new_max = [&](float tmax) __attribute__((always_inline)) {       // of a tile: both halves of the wave hold keys of the same row
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
    const float mt = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * a.scale_log2;
    if (__builtin_amdgcn_ballot_w64(mt > m_run)) {
      const float m_new = fmaxf(m_run, mt);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;       // (nothing visible yet)
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);    // m_run = -inf -> 0
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
      m_run = m_new;
      neg_m = -m_use;
    }
  };
  // CUR: S holds tile kt's masked scores; NEXT: the wave works in tile kt + 1 too; ODD: kt is odd (one wave a row: the second tile of a step)
  auto step = [&](int kt, auto CURT, auto NEXTT, auto ODDT, Scores& S, Scores& SN) __attribute__((always_inline)) {
    constexpr bool CUR = decltype(CURT)::value, NEXT = decltype(NEXTT)::value, ODD = decltype(ODDT)::value;
    constexpr int KOFF = KG == 1 && !ODD && CUR ? TILEB : 0, VOFF = KG == 1 && ODD ? TILEB : 0;      // (without CUR: the first tile of a step)
    constexpr bool COPIES = SLOTS > 1 && CUR && (TPS == 1 || !ODD);        // the first tile of a step: the next one's copies, spread (64 of them at once hold up every wave)
    constexpr int NC = 4 * PPT, NM = NQK + NPV;
    static_assert(!COPIES || (NM >= NC && copies_before(NM, NM, NC) == NC), "every copy once");
    auto copy_behind = [&](auto I) __attribute__((always_inline)) {
      constexpr int c = copies_before(decltype(I)::value, NM, NC);
      if constexpr (copies_before(decltype(I)::value + 1, NM, NC) > c) copy_ahead(kt, c);
    };
    if constexpr (COPIES && !NEXT)
#pragma unroll
      for (int c = 0; c < 4 * PPT; ++c) copy_ahead(kt, c);
    if constexpr (NEXT && CUR && (KG == 2 || ODD)) {             // tile kt + 1 is in the ring's other half
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) k_rd[ks] ^= HALF;
    }
    float ps0 = 0.f, ps1 = 0.f, nm = neg_m;
    asm volatile("" : "+v"(nm));             // (the exponents of all forms of a step would be formed in front of the branch between them)
    u32x4 pf[2 * KT];
    auto weights = [&](auto FROM, auto TO) __attribute__((always_inline)) {
      static_for<decltype(FROM)::value / 2, decltype(TO)::value / 2>([&](auto E) __attribute__((always_inline)) {
        constexpr int e = 2 * decltype(E)::value;
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e >> 4][e & 15], a.scale_log2, nm));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e >> 4][(e & 15) + 1], a.scale_log2, nm));
        ps0 += p0;
        ps1 += p1;
        const v2 pair = {from_f32<T>(p0), from_f32<T>(p1)};
        pf[e >> 3][(e & 7) >> 1] = __builtin_bit_cast(unsigned, pair);
        // (formed HERE: the compiler would sink all of it behind the next branch, where the matrix pipe has nothing to do)
        asm volatile("" : "+v"(pf[e >> 3][(e & 7) >> 1]), "+v"(ps0), "+v"(ps1));
      });
    };
    auto largest = [&](auto FROM, auto TO, float m) __attribute__((always_inline)) {
      static_for<decltype(FROM)::value, decltype(TO)::value>([&](auto E) __attribute__((always_inline)) {
        constexpr int e = 2 * decltype(E)::value;
        m = fmaxf(fmaxf(m, SN[e >> 4][e & 15]), SN[e >> 4][(e & 15) + 1]);
      });
      return m;
    };
    v4 vlo[2][DT], vhi[2][DT];
    auto read_v = [&](int s_, int dt) __attribute__((always_inline)) {
      // element j of this lane is key row 16s + 8(j>>2) + 4hh + (j&3) of the tile
      const lds_u8* at = lds_at(FEW ? v_rd[0] ^ (unsigned)(dt << 6) : v_rd[FEW ? 0 : dt]) + VOFF;
      vlo[s_ & 1][dt] = Frag<T>::tr_read(at + s_ * (16 * ROWB));
      vhi[s_ & 1][dt] = Frag<T>::tr_read(at + s_ * (16 * ROWB) + 8 * ROWB);
    };
    using std::integral_constant;
    if constexpr (NEXT) {
      v8 kf[NQK];
      auto read_k = [&](int i) __attribute__((always_inline)) { kf[i] = Frag<T>::row_read(lds_at(FEW ? k_rd[0] ^ (unsigned)(32 * (i % KS)) : k_rd[FEW ? 0 : i % KS]) + KOFF + (i / KS) * (32 * ROWB)); };
#pragma unroll
      for (int i = 0; i < KAHEAD; ++i) read_k(i);
      if constexpr (CUR) weights(integral_constant<int, 0>{}, integral_constant<int, LEAD>{});
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, NQK>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        if constexpr (i + KAHEAD < NQK) read_k(i + KAHEAD);
        if constexpr (CUR && i >= NQK - DT) read_v(0, i - (NQK - DT));
        if constexpr (i % KS == 0)
#pragma unroll
          for (int j = 0; j < 16; ++j) SN[i / KS][j] = 0.f;
        SN[i / KS] = Frag<T>::mfma(kf[i], qf[i % KS], SN[i / KS]);
        if constexpr (CUR && COPIES) copy_behind(I);
        if constexpr (CUR) weights(integral_constant<int, LEAD + 2 * ((NE1 - LEAD) / 2 * i / NQK)>{}, integral_constant<int, LEAD + 2 * ((NE1 - LEAD) / 2 * (i + 1) / NQK)>{});
        __builtin_amdgcn_sched_barrier(0);
      });
      mask(kt + 1, SN);
    } else {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) read_v(0, dt);
      weights(integral_constant<int, 0>{}, integral_constant<int, NE1>{});
    }
    float tmax = -INFINITY;
    if constexpr (CUR) {
      __builtin_amdgcn_s_setprio(1);            // P.V first where both waves of a SIMD want the matrix pipe (16 384 tokens, 40 heads: 2 467 -> 2 445 us)
      constexpr int NP1 = NPV - DT;             // (the last k-step needs all of them)
      static_assert(NE1 >= 8 && NE1 % 2 == 0, "the first k-step's weights come first");
      static_for<0, NPV>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value, s_ = i / DT, dt = i % DT;
        if constexpr (s_ + 1 < 2 * KT) read_v(s_ + 1, dt);
        v8 vf;
#pragma unroll
        for (int j = 0; j < 4; ++j) { vf[j] = vlo[s_ & 1][dt][j]; vf[4 + j] = vhi[s_ & 1][dt][j]; }
        oacc[dt] = Frag<T>::mfma(vf, __builtin_bit_cast(v8, pf[s_]), oacc[dt]);
        if constexpr (i < NP1) weights(integral_constant<int, NE1 + 2 * ((NE - NE1) / 2 * i / NP1)>{}, integral_constant<int, NE1 + 2 * ((NE - NE1) / 2 * (i + 1) / NP1)>{});
        if constexpr (NEXT && COPIES) copy_behind(integral_constant<int, NQK + i>{});
        constexpr int M0 = 2;                   // (the scores' last MFMA ends behind the first of these)
        if constexpr (NEXT && i >= M0) tmax = largest(integral_constant<int, NE / 2 * (i - M0) / (NPV - M0)>{}, integral_constant<int, NE / 2 * (i + 1 - M0) / (NPV - M0)>{}, tmax);
        __builtin_amdgcn_sched_barrier(0);
      });
      __builtin_amdgcn_s_setprio(0);
      l_run += ps0 + ps1;
    } else {
      tmax = largest(integral_constant<int, 0>{}, integral_constant<int, NE / 2>{}, tmax);
    }
    if constexpr (CUR && (KG == 2 || ODD)) {                    // tile kt + 1's V is in the other half
#pragma unroll
      for (int dt = 0; dt < NV; ++dt) v_rd[dt] ^= HALF;
    }
    if constexpr (NEXT) new_max(tmax);
  };
  // The step that starts with this wave's tile kt: its V and the K of the tiles behind each are there for every wave, and nobody reads the other two places of a ring
  // any more, which the next step's copies take.  (One barrier for two tiles.)
  auto turn = [&](int kt, bool idle) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (SLOTS > 1 && idle)
#pragma unroll
      for (int c = 0; c < 4 * PPT; ++c) copy_ahead(kt, c);
  };
  {
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    int kt = 0;
    // (a run starts with the first tile of a step)
    const int run2 = TPS == 2 ? win_from & ~1 : own(win_from);
    const bool one = !WIN || run2 <= own(keep_to);                  // nothing left out: one run of tiles
#pragma unroll 1
    for (int run = one ? 1 : 0; run < 2; ++run) {
      const int from = one || !run ? 0 : run2, to = own(one || run ? n_seen : keep_to);
      if (from >= to) continue;
      for (; kt + TPS < from; kt += TPS) turn(kt, true);
      if (kt < from) { turn(kt, true); kt += TPS; }
      set_reads(HALF & (unsigned)-(int)((from * KG >> 1) & 1));
      step(from - 1, no, yes, no, s1, s0);
      if constexpr (SLOTS > 1) {
#pragma unroll 1
        for (; kt + 2 < to; kt += 2) {
          turn(kt, false);
          step(kt, yes, yes, no, s0, s1);
          if (TPS == 1) turn(kt + 1, false);
          step(kt + 1, yes, yes, yes, s1, s0);
        }
      }
      turn(kt, false);
      if (SLOTS > 1 && kt + 1 < to) {
        step(kt, yes, yes, no, s0, s1);
        if (TPS == 1) turn(kt + 1, false);
        step(kt + 1, yes, no, yes, s1, s0);
        kt += 2;
      } else {
        step(kt, yes, no, no, s0, s1);
        kt += TPS;
      }
    }
    for (; kt < nown; kt += TPS) turn(kt, true);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  }

  // ---- epilogue: normalise and store O[q][d] ----
  const int le = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));      // the lane, anew: what hangs on it would be carried through the loop and spilled
  const int hh_e = le >> 5, qrow_e = q0 + (le & 31);
  float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  // KG 2: the two waves of a row meet over the ring; the first keeps the first half of the d-tiles, the second the rest
  constexpr int DH = (DT + 1) / 2;
  if constexpr (KG == 2) {
    f32x4* const xo = (f32x4*)fa_smem;                    // [wave][d-tile of the partner][4][lane]
    float* const xm = (float*)(fa_smem + NW * DH * 4 * 64 * 16);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      if ((dt < DH) == (grp == 1)) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          xo[((wave * DH + (dt < DH ? dt : dt - DH)) * 4 + g) * 64 + le] = f32x4{oacc[dt][4 * g], oacc[dt][4 * g + 1], oacc[dt][4 * g + 2], oacc[dt][4 * g + 3]};
      }
    xm[(wave * 2 + 0) * 64 + le] = m_run;
    xm[(wave * 2 + 1) * 64 + le] = l_tot;
    __syncthreads();
    const int other = wave ^ (NW / 2);
    const float m_o = xm[(other * 2 + 0) * 64 + le], l_o = xm[(other * 2 + 1) * 64 + le], m_all = fmaxf(m_run, m_o);
    const float f = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_all), f_o = m_o == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_o - m_all);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      if ((dt < DH) == (grp == 0)) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = xo[((other * DH + (dt < DH ? dt : dt - DH)) * 4 + g) * 64 + le];
#pragma unroll
          for (int j = 0; j < 4; ++j) oacc[dt][4 * g + j] = oacc[dt][4 * g + j] * f + v[j] * f_o;
        }
      }
    l_tot = l_tot * f + l_o * f_o;
    m_run = m_all;
  }
  if (a.sink) l_tot += __builtin_amdgcn_exp2f(a.sink[h] * 1.4426950408889634f - m_run);      // (not scaled; inf: the keys weigh nothing)
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (qrow_e < Lq) {
    T* op = (T*)a.o + (WIN ? 0 : (int64_t)b * a.osb) + (row0 + qrow_e) * a.osl + (int64_t)h * a.osh;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d0 = dt * 32 + 8 * g + 4 * hh_e;
        if (KG == 2 && (dt < DH) != (grp == 0)) continue;
        if (d0 < a.Dv) {
          v4 pk;
          if constexpr (WIN) {
            if (a.gate) {
              const v4 gt = *(const v4*)((const T*)a.gate + (row0 + qrow_e) * a.gsl + (int64_t)h * a.gsh + d0);
#pragma unroll
              for (int j = 0; j < 4; ++j) oacc[dt][4 * g + j] *= sigmoid_f((float)gt[j]);
            }
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) pk[j] = from_f32<T>(oacc[dt][4 * g + j] * inv);
          *(v4*)(op + d0) = pk;
        }
      }
    if (!WIN && a.lse && hh_e == 0 && grp == 0) {
      const float lse = l_tot > 0.f ? (m_run * 0.6931471805599453f + logf(l_tot)) : -INFINITY;
      a.lse[((int64_t)b * a.Hq + h) * Lq + qrow_e] = lse;
    }
  }
}


// -DTV_FA_STAMP (dev): waves 0 and 4 of work-group 0 of the streaming kernel sum the cycles of each phase
// of tile kt (s_memtime): g_fa_stamps[wave/4][kt < 16][phase < 8]; tv_fa_debug_stamps() copies them out.
#ifdef TV_FA_STAMP
__device__ unsigned long long g_fa_stamps[2 * 16 * 8];
#define FSTAMP(ph) do { if (st_on) { const unsigned long long n__ = clock64(); if (lane == 0) st_acc[((wave >> 2) * 16 + (kt < 16 ? kt : 15)) * 8 + ph] += n__ - st_last; st_last = n__; } } while (0)
#else
#define FSTAMP(ph) do {} while (0)
#endif

// Many short sequences (ViT frames: 729 tokens = 8 key tiles per query block): a work-group that
// handles ONE query block spends a third of its life outside the tile loop — waiting for Q and the
// first two K/V tiles, zeroing LDS, storing O — and at 147 KiB of LDS nothing else is resident on
// the CU to cover that (measured: 27.9 us per work-group of which 8 x 2.2 us in the loop).  This
// kernel keeps the work-group and STREAMS query blocks through it: the K/V ring never drains — the
// copies of the next block's first two tiles are issued under the last two tiles of the current
// one, its Q fragments are loaded under the last tile — and the O stores of a block complete under
// the first tile of the next.  Non-causal, >= 2 key tiles.  Grid: 8 x (work-groups per XCD); the
// work-groups of XCD x walk slots x*... of that XCD's contiguous range of (batch, head) pairs, so the
// query blocks that share K / V still meet in one L2 at about the same time.
// ONES (head_dim a multiple of 8 and < 32 DT: the ViT's 72): the row sums of P come out of the P.V MFMAs.  The pad chunks
// of the rings are written ONCE (zeros; V column head_dim = 1.0) and the copy lanes that would land on them are switched
// off (a constant EXEC mask per wave around each piece: the swizzle depends on row & 15 only), so O^T row head_dim
// accumulates sum_k bf16(P[q][k]) — rescaled by alpha with the rest of the tile — and the per-tile adds for l go away.
// l is then the sum of the ROUNDED weights, the ones the output was built from.
template <typename T, int KS, int DT, int KT, bool ONES>
__global__ __launch_bounds__(512) void flash_fwd_stream_kernel(AttnArgs a) {
  constexpr int NW = 8;
  constexpr int FA_KB = 32 * KT;
  constexpr int NPK = FA_KB / 4;
  typedef typename Frag<T>::v8 v8;
  typedef typename Frag<T>::v4 v4;
  constexpr int QB = NW * FA_QW;
  constexpr int ROWB = 256;
  constexpr int TILEB = FA_KB * ROWB;
  constexpr int NS = 3;
  constexpr int PPW = 2 * NPK / NW;
  static_assert(2 * NPK % NW == 0, "pieces must divide over the waves");
  extern __shared__ __attribute__((aligned(16))) unsigned char fa_smem[];
  const unsigned sK_off = (unsigned)(uintptr_t)(lds_u8*)fa_smem, sV_off = sK_off + NS * TILEB;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 31, hh = lane >> 5;
  const int D = a.D;
  const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
  const int nslots = a.ppx * a.nqb, npairs = a.nb * a.Hq;
  int slot = blockIdx.x >> 3;
  int pair = xcd * a.ppx + slot / a.nqb, qblk = slot % a.nqb;
  if (slot >= nslots || pair >= npairs) return;
  const int gq = a.Hq / a.Hkv;
  auto k_of = [&](int pr) { return (const T*)a.k + (int64_t)(pr / a.Hq) * a.ksb + (int64_t)((pr % a.Hq) / gq) * a.ksh; };
  auto v_of = [&](int pr) { return (const T*)a.v + (int64_t)(pr / a.Hq) * a.vsb + (int64_t)((pr % a.Hq) / gq) * a.vsh; };
  // Q^T fragments (B operand): lane (r,hh) holds Q[qrow][16ks + 8hh + j]
  // untracked loads (gload16_async) + a finishing step behind the counted wait that covers them
  auto load_q = [&](int pr, int qb, u32x4 (&raw)[KS]) {
    const T* qp = (const T*)a.q + (int64_t)(pr / a.Hq) * a.qsb + (int64_t)(pr % a.Hq) * a.qsh;
    const int qrow = qb * QB + wave * FA_QW + r;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = ks * 16 + hh * 8;
      raw[ks] = gload16_async((qrow < a.Lq && d0 < D) ? qp + (int64_t)qrow * a.qsl + d0 : qp);
    }
  };
  auto finish_q = [&](int qb, u32x4 (&raw)[KS], v8 (&qf)[KS]) {
    const int qrow = qb * QB + wave * FA_QW + r;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      settle(raw[ks]);
      const v8 z = {};
      qf[ks] = (qrow < a.Lq && ks * 16 + hh * 8 < D) ? __builtin_bit_cast(v8, raw[ks]) : z;
    }
  };
  v8 qf[KS];
  u32x4 qn[KS];
  load_q(pair, qblk, qn);

  // ---- DMA pieces of this wave: K pieces wave + NW i (4 key rows each, i < KPW), as many of V; lane l
  // carries row 4 piece + l/16, LDS slot l%16 (source chunk = slot ^ swizzle).  Lanes whose chunk lies
  // past head_dim re-fetch chunk 0 of their row instead of being masked off: the pad slots then hold
  // finite copies of real values — K pad columns meet Q columns that are exact zeros, V pad columns
  // feed output rows that are never stored — and the issue path needs no EXEC juggling: per piece one
  // scalar add for M0 and the copy itself (the masked, per-piece-addressed form cost ~300 cycles a
  // piece and paced the whole QK^T phase: 2 100 cycles for 480 cycles of MFMA) ----
  static_assert(NPK % NW == 0, "K pieces must divide over the waves");
  constexpr int KPW = NPK / NW;
  const int dchunks = D / 8;
  int p_row[KPW];
  unsigned offK[KPW], offV[KPW], coK[KPW], coV[KPW];
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int row = 4 * (wave + NW * i) + (lane >> 4);
    int ck = (lane & 15) ^ (row & 15), cv = (lane & 15) ^ (4 * (row & 3));
    ck = ck < dchunks ? ck : 0;
    cv = cv < dchunks ? cv : 0;
    p_row[i] = row;
    coK[i] = (unsigned)(ck * 8 * (int)sizeof(T));
    coV[i] = (unsigned)(cv * 8 * (int)sizeof(T));
    offK[i] = (unsigned)(row * (int)a.ksl * (int)sizeof(T)) + coK[i];
    offV[i] = (unsigned)(row * (int)a.vsl * (int)sizeof(T)) + coV[i];
  }
  const unsigned m0_wave = (unsigned)(wave * 1024);
  // ONES: lanes whose slot is a pad chunk stay out of the copies (same lanes for every piece of a wave)
  const unsigned long long liveK = __builtin_amdgcn_ballot_w64(((lane & 15) ^ ((4 * wave + (lane >> 4)) & 15)) < dchunks);
  const unsigned long long liveV = __builtin_amdgcn_ballot_w64(((lane & 15) ^ (4 * ((lane >> 4) & 3))) < dchunks);
  if constexpr (ONES) {
    // pad chunks of every ring row: K zeros (they meet Q columns that are zero, but must be finite), V zeros and the
    // ones column.  16 bytes a chunk; rows are 256 bytes, chunk c of row `row` lives in slot c ^ swizzle(row).
    const v8 one_first = [] { v8 z = {}; z[0] = from_f32<T>(1.f); return z; }();
    const v8 zero8 = {};
    for (int i = tid; i < NS * FA_KB * 16; i += 512) {
      const int row = i >> 4, c = i & 15;
      if (c >= dchunks) {
        *(v8*)(fa_smem + row * ROWB + ((c ^ (row & 15)) << 4)) = zero8;
        *(v8*)(fa_smem + NS * TILEB + row * ROWB + ((c ^ (4 * (row & 3))) << 4)) = c == dchunks ? one_first : zero8;
      }
    }
    __syncthreads();
  }
  // tile `kt` of the sequence at kpx / vpx into ring stage `stage`: piece j (0..PPW-1; K first)
  struct TileCopy { const unsigned char *tk, *tv; unsigned mk; int left; };
  auto tile_copy = [&](const T* kpx, const T* vpx, int kt, int stage) {
    TileCopy c;
    c.tk = (const unsigned char*)(kpx + (int64_t)kt * FA_KB * a.ksl);
    c.tv = (const unsigned char*)(vpx + (int64_t)kt * FA_KB * a.vsl);
    c.mk = sK_off + (unsigned)(stage * TILEB) + m0_wave;
    c.left = a.Lk - kt * FA_KB;                 // rows of this tile that exist
    return c;
  };
  auto issue_piece = [&](const TileCopy& c, int j) {
    const bool isK = j < KPW;                   // compile-time after unrolling
    const int i = isK ? j : j - KPW;
    unsigned off = isK ? offK[i] : offV[i];
    if (c.left < FA_KB) {                       // last tile: rows past the end repeat the last key (masked later)
      const int rr = min(p_row[i], c.left - 1);
      off = (unsigned)(rr * (int)(isK ? a.ksl : a.vsl) * (int)sizeof(T)) + (isK ? coK[i] : coV[i]);
    }
    if constexpr (ONES)
      glds16_lanes(isK ? c.tk : c.tv, off, c.mk + (unsigned)(i * NW * 1024) + (isK ? 0u : (unsigned)(NS * TILEB)),
                         isK ? liveK : liveV);
    else
      ssdk::glds16(isK ? c.tk : c.tv, off, c.mk + (unsigned)(i * NW * 1024) + (isK ? 0u : (unsigned)(NS * TILEB)));
  };

  int k_rd[KS];
  const int kz = (hh ^ (r & 15)) << 4;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_rd[ks] = r * ROWB + ((32 * ks) ^ kz);
  const int q4 = (lane & 15) >> 2, p4 = lane & 3;
  int v_rd[DT];
  {
    const int cc = 2 * ((lane >> 4) & 1) + (p4 >> 1);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      v_rd[dt] = (4 * hh + q4) * ROWB + ((4 * (dt ^ q4) + cc) << 4) + (p4 & 1) * 8;
  }

  const int ntiles = (a.Lk + FA_KB - 1) / FA_KB;       // >= 2 (launcher)
  const T* kp = k_of(pair);
  const T* vp = v_of(pair);
  {
    const TileCopy c0 = tile_copy(kp, vp, 0, 0), c1 = tile_copy(kp, vp, 1, 1);
#pragma unroll
    for (int j = 0; j < PPW; ++j) issue_piece(c0, j);
#pragma unroll
    for (int j = 0; j < PPW; ++j) issue_piece(c1, j);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW) : "memory");
  __builtin_amdgcn_s_barrier();
  finish_q(qblk, qn, qf);

  // the second-dispatched half of the work-group loses every VALU arbitration to the older half (priority, then
  // age): one static priority bump for it, no per-phase flips (-0.8 % here; the causal and fp8 kernels measured
  // 0.5 - 1 % SLOWER with it and do not have it)
  if (wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
  int stage = 0;                   // ring stage of the current tile
#ifdef TV_FA_STAMP
  const bool st_on = blockIdx.x == 0 && (wave == 0 || wave == 4);
  __shared__ unsigned long long st_acc[2 * 16 * 8];
  if (tid < 256) st_acc[tid] = 0;
  __syncthreads();
  unsigned long long st_last = clock64();
#endif
  for (;;) {
    const int slot_n = slot + step;
    const int pair_n = xcd * a.ppx + slot_n / a.nqb, qblk_n = slot_n % a.nqb;
    const bool has_next = slot_n < nslots && pair_n < npairs;
    const T* kp_n = has_next ? k_of(pair_n) : kp;
    const T* vp_n = has_next ? v_of(pair_n) : vp;

    f32x16 oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    for (int kt = 0; kt < ntiles; ++kt) {
      const int kbase = kt * FA_KB;
      // the copy that goes out under this tile: two tiles on, in this block or the next one
      const bool wrap = kt + 2 >= ntiles;
      const bool ahead = !wrap || has_next;
      const T* pk = wrap ? kp_n : kp;
      const T* pv = wrap ? vp_n : vp;
      const int pf_kt = wrap ? kt + 2 - ntiles : kt + 2;
      const int pf_stage = stage == 0 ? 2 : stage - 1;
      const TileCopy pf = tile_copy(pk, pv, pf_kt, pf_stage);
      if (kt == ntiles - 1 && has_next) load_q(pair_n, qblk_n, qn);   // older than this tile's copies
      const unsigned stage_off = (unsigned)(stage * TILEB);
      const unsigned cK = sK_off + stage_off, cV = sV_off + stage_off;

      auto tile_body = [&](auto nt_c) __attribute__((always_inline)) {
      constexpr int NT = decltype(nt_c)::value;        // live 32-key sub-tiles of this tile
      f32x16 sacc[NT];
      v8 kf[NT][KS];
      unsigned kb[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kb[ks] = cK + (unsigned)k_rd[ks];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[t][ks] = Frag<T>::row_read(lds_at(kb[ks]) + t * (32 * ROWB));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sacc[t][i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          sacc[t] = Frag<T>::mfma(kf[t][ks], qf[ks], sacc[t]);
          // the copies of tile kt+2 go out between the MFMAs (placing them between the exponentials
          // of the softmax instead measured the same)
          constexpr int every = (NT * KS) / PPW > 0 ? (NT * KS) / PPW : 1;
          const int idx = t * KS + ks;
          if (ahead && idx % every == 0 && idx / every < PPW) issue_piece(pf, idx / every);
        }
      }
      if (ahead) {
#pragma unroll
        for (int i = (NT * KS) / ((NT * KS) / PPW > 0 ? (NT * KS) / PPW : 1); i < PPW; ++i)
          issue_piece(pf, i);
      }
      FSTAMP(0);
      typedef float f32x2 __attribute__((ext_vector_type(2)));
      if (kbase + FA_KB > a.Lk) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = kbase + t * 32 + (i & 3) + 8 * (i >> 2) + 4 * hh;
            sacc[t][i] = key < a.Lk ? sacc[t][i] : -INFINITY;
          }
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += 2) tmax = fmaxf(fmaxf(tmax, sacc[t][i]), sacc[t][i + 1]);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m_run, tmax * a.scale_log2);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
      const f32x2 sc2 = {a.scale_log2, a.scale_log2}, nm2 = {-m_use, -m_use};
      f32x2 ps2 = {0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const f32x2 e = __builtin_elementwise_fma(f32x2{sacc[t][i], sacc[t][i + 1]}, sc2, nm2);
          const f32x2 pp = {__builtin_amdgcn_exp2f(e[0]), __builtin_amdgcn_exp2f(e[1])};
          sacc[t][i] = pp[0];
          sacc[t][i + 1] = pp[1];
          if constexpr (!ONES) ps2 += pp;
        }
      if constexpr (!ONES) l_run = l_run * alpha + (ps2[0] + ps2[1]);
      if (__builtin_amdgcn_ballot_w64(m_new > m_run)) {
        const f32x2 al2 = {alpha, alpha};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            const f32x2 v = f32x2{oacc[dt][i], oacc[dt][i + 1]} * al2;
            oacc[dt][i] = v[0];
            oacc[dt][i + 1] = v[1];
          }
      }
      m_run = m_new;
      FSTAMP(1);
      {
        unsigned vb[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vb[dt] = cV + (unsigned)v_rd[dt];
        auto read_v = [&](int s_, v4 (&lo)[DT], v4 (&hi)[DT]) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            lo[dt] = Frag<T>::tr_read(lds_at(vb[dt]) + s_ * (16 * ROWB));
            hi[dt] = Frag<T>::tr_read(lds_at(vb[dt]) + s_ * (16 * ROWB) + 8 * ROWB);
          }
        };
        v4 vlo[2][DT], vhi[2][DT];
        read_v(0, vlo[0], vhi[0]);
#pragma unroll
        for (int s_ = 0; s_ < 2 * NT; ++s_) {
          if (s_ < 2 * NT - 1) read_v(s_ + 1, vlo[(s_ + 1) & 1], vhi[(s_ + 1) & 1]);
          const int t = s_ >> 1, rb = (s_ & 1) * 8;
          v8 pf;
#pragma unroll
          for (int j = 0; j < 8; ++j) pf[j] = from_f32<T>(sacc[t][rb + j]);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            v8 vf;
#pragma unroll
            for (int j = 0; j < 4; ++j) { vf[j] = vlo[s_ & 1][dt][j]; vf[4 + j] = vhi[s_ & 1][dt][j]; }
            oacc[dt] = Frag<T>::mfma(vf, pf, oacc[dt]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      };
      // a frame's last tile is rarely full (729 keys = 7 x 96 + 57): sub-tiles that hold no key at all are left out of
      // the products, the exponentials and the V reads (the copies still bring the whole tile: the ring's shape is fixed)
      const int live_keys = a.Lk - kbase;
      // (not at 6 k-steps: three bodies beside 24 more fragment registers do not fit the 256)
      if (KT < 3 || KS > 5 || live_keys > 64 || a.notrim) tile_body(std::integral_constant<int, KT>{});
      else if (live_keys > 32) tile_body(std::integral_constant<int, (KT > 2 ? 2 : KT)>{});
      else tile_body(std::integral_constant<int, 1>{});
      FSTAMP(2);
      // the next tile (copied an iteration ago) must have landed; this iteration's copies stay in flight
      if (ahead) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      FSTAMP(3);
      __builtin_amdgcn_s_barrier();
      FSTAMP(4);
      stage = stage == NS - 1 ? 0 : stage + 1;
    }

    // ---- normalise and store O[q][d] of this block; the stores complete under the next block's first tile ----
    {
      const int h = pair % a.Hq, b = pair / a.Hq;
      const int qrow = qblk * QB + wave * FA_QW + r;
      float l_tot;
      if constexpr (ONES) {
        // O^T row head_dim of query r: d-tile DT - 1, local row D - 32 (DT - 1) (a multiple of 8: element 4 (row / 8) of
        // the lane with hh = 0)
        const int rl8 = (D - 32 * (DT - 1)) >> 3;
        float lv = 0.f;
#pragma unroll
        for (int g = 0; g < 4; ++g) lv = g == rl8 ? oacc[DT - 1][4 * g] : lv;
        const float lo = __shfl_xor(lv, 32, 64);
        l_tot = hh ? lo : lv;
      } else {
        l_tot = l_run + __shfl_xor(l_run, 32, 64);
      }
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
      // A lane holds 4 output columns (8 bytes) per (d-tile, group g): columns 32 dt + 8 g + 4 hh .. + 3.  The halves
      // hh = 0 / 1 of a lane pair (r, r + 32) own the two halves of 8 consecutive columns, so one
      // v_permlane32_swap per dword gives each lane 16 contiguous bytes (groups g, g + 1 -> the lower lane
      // stores columns 16 gp .. + 7, the upper lane the next 8): half the store instructions — the epilogue of
      // a block is store-ISSUE bound.  Needs 16-byte aligned rows (a.o16); the last lone group stays 8 bytes.
      typedef unsigned u32x2s __attribute__((ext_vector_type(2)));
      typedef unsigned u32x4s __attribute__((ext_vector_type(4)));
      T* op = (T*)a.o + (int64_t)b * a.osb + (int64_t)min(qrow, a.Lq - 1) * a.osl + (int64_t)h * a.osh;
      const bool rowok = qrow < a.Lq;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          const int d_lo = dt * 32 + 16 * gp;          // first column of the pair of groups
          if (d_lo >= D) continue;
          v4 pa, pb;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            pa[j] = from_f32<T>(oacc[dt][4 * (2 * gp) + j] * inv);
            pb[j] = from_f32<T>(oacc[dt][4 * (2 * gp + 1) + j] * inv);
          }
          if (a.o16 && d_lo + 8 < D) {                 // (wave-uniform)
            const u32x2s ua = __builtin_bit_cast(u32x2s, pa), ub = __builtin_bit_cast(u32x2s, pb);
            const auto s0 = __builtin_amdgcn_permlane32_swap(ua[0], ub[0], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(ua[1], ub[1], false, false);
            const u32x4s w = {s0[0], s1[0], s0[1], s1[1]};
            if (rowok) *(u32x4s*)(op + d_lo + 8 * hh) = w;
          } else {
            if (rowok) *(v4*)(op + d_lo + 4 * hh) = pa;
            if (rowok && d_lo + 8 + 4 * hh < D) *(v4*)(op + d_lo + 8 + 4 * hh) = pb;
          }
        }
      if (rowok) {
        if (a.lse && hh == 0) {
          const float lse = l_tot > 0.f ? (m_run * 0.6931471805599453f + logf(l_tot)) : -INFINITY;
          a.lse[((int64_t)b * a.Hq + h) * a.Lq + qrow] = lse;
        }
      }
    }
    { const int kt = 15; FSTAMP(5); (void)kt; }
    if (!has_next) break;
    slot = slot_n; pair = pair_n; qblk = qblk_n; kp = kp_n; vp = vp_n;
    finish_q(qblk, qn, qf);        // loaded under the last tile, older than the copies its wait left in flight
  }
#ifdef TV_FA_STAMP
  __syncthreads();
  if (blockIdx.x == 0 && tid < 256) g_fa_stamps[tid] = st_acc[tid];
#endif
}


#include "attention_vit.hpp"

std::atomic<int> g_fa_variant{[] { const char* v = getenv("TV_FA_W64"); return v ? atoi(v) : 0; }()};

// When the last of a grid's work-groups ends, one of them a compute unit at a time, each starting where a unit is free first: runs of equal ones in grid order.  Its
// unit of time is a quarter of a step of 128 keys by two waves a row, which 96 keys by one wave take as well; a block's start and end take 10.
struct Dealt {
  struct Run { int64_t end; int n; } runs[512];     // (every run is a compute unit or more: never more runs than those)
  int size = 1;
  int64_t last = 0;
  Dealt() { runs[0] = {0, std::max(1, std::min(tv_cu_count(), 512))}; }
  void add(int64_t cost, int64_t n) {
    const auto later = [](const Run& a, const Run& b) { return a.end > b.end; };
    while (n > 0) {
      std::pop_heap(runs, runs + size, later);
      Run& first = runs[size - 1];
      const Run taken{first.end + cost, (int)std::min<int64_t>(first.n, n)};
      n -= taken.n;
      last = std::max(last, taken.end);
      if ((first.n -= taken.n) == 0) first = taken;
      else { std::push_heap(runs, runs + size, later); runs[size++] = taken; }
      std::push_heap(runs, runs + size, later);
    }
  }
};
// Blocks of 256 rows are at most a round (their longest ends last): whether those of 128 rows, more than one, end before .94 of it, and before .99 at head dim 128, where a
// step of one wave takes a little more than the estimate (16 heads, 4 096 rows against 5 120 keys: 159 | 145 us, estimated alike)
bool dealt_out_pays(const Dealt& two, int64_t one, bool wide) { return two.last * 100 < one * (wide ? 99 : 94); }

// Whether two waves share 32 query rows (KG 2): up to 128 rows, while 128-row blocks are one round of the compute units (us, one wave | two: 40 heads x 128, 700 tokens
// 24.9 | 18.6, 28 x 1 100 33.8 | 24.3; 64 wide, 40 x 700 18.5 | 13.3), and for more of them where causal blocks grow from nothing and the short ones, dealt out last,
// fill up the long ones' time (40 x 1 400: 42.1 | 38.8, 28 x 2 000: 56.6 | 47.0; not 40 x 2 000, 320 blocks of 256: 60.3 | 67.1; nor whole rows).
// The line is the estimate above: over 707 shapes of 130 to 4 000 rows (head dims 64, 80, 128; 4 to 160 pairs; triangles, triangles behind earlier keys, whole rows) what it
// takes is .5 % slower in the mean than the better form of each; one wave always is 20 % slower, two 4 %.
bool two_waves_a_row(int Lq, int Lk, int64_t pairs, bool causal, bool wide) {
  const int cus = tv_cu_count(), rows = (Lq + 127) / 128;
  if (Lq <= 128 || rows * pairs <= cus) return true;
  if (!causal || Lk - Lq > Lq / 4 || (Lq + 255) / 256 * pairs > cus) return false;
  Dealt two;
  for (int q = rows; q > 0; --q) two.add(10 + 4 * ((std::max<int64_t>(0, std::min<int64_t>(Lk, q * 128ll + Lk - Lq)) + 127) / 128), pairs);
  return dealt_out_pays(two, 10 + 4 * ((Lk + 95ll) / 96), wide);
}
// ... but not for short rows whose keys are one tile of 96: four waves, no ring, a third of the LDS, so that several such work-groups run on a compute unit; by head and
// batch entry, without a division (us, two waves a row | this, causal: 16 heads of 64: 1 x 1 5.7 | 5.5, 64 x 64 6.2 | 5.8, 96 x 96 7.0 | 6.1; of 128: 8.2 | 6.6, 9.6 | 7.3; 4 000 pairs
// 64 wide, 33 x 33 83 | 35, 128 x 96 107 | 46; 128 wide, 111 | 41, 173 | 84; the worst of 80 forms, 16 heads of 64, 64 x 64 without a mask: 5.7 | 5.9).
bool one_tile(int Lk, int tile) { return Lk <= tile; }

template <typename T, int KS, int DT>
int launch_fa_d(const AttnArgs& a, int B, hipStream_t st) {
  constexpr int KT = FA_KT;
  constexpr int lds = 2 * 3 * 32 * KT * 256;   // K and V rings: 3 stages x 32 KT rows x 256 B
  constexpr int lds1 = fa_lds(KT), lds2 = fa_lds(2);
  hipError_t e;
  const int64_t all = (int64_t)a.Hq * B;
  const int nqb = (a.Lq + 255) / 256;
  static const int xcd_ = [] { const char* v = getenv("TV_FA_XCD"); return v ? atoi(v) : 1; }();
  const bool frames = a.Lq > 128 && xcd_ && !a.causal && nqb <= 8 && all >= 64;
  if (a.Lq <= 128 && one_tile(a.Lk, 32 * KT) && B <= 65535 && a.Hq <= 65535) {
    e = hipFuncSetAttribute((const void*)flash_fwd_kernel<T, KS, DT, 4, KT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds1);
    if (e == hipSuccess) flash_fwd_kernel<T, KS, DT, 4, KT><<<dim3(1, (unsigned)a.Hq, (unsigned)B), 256, lds1, st>>>(a, NoSeqs{});
  } else if (!frames && two_waves_a_row(a.Lq, a.Lk, all, a.causal, KS > 6)) {
    e = hipFuncSetAttribute((const void*)flash_fwd_kernel<T, KS, DT, 8, 2, false, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, lds2);
    if (e == hipSuccess) flash_fwd_kernel<T, KS, DT, 8, 2, false, 2><<<dim3((unsigned)((a.Lq + 127) / 128 * all)), 512, lds2, st>>>(a, NoSeqs{});
  } else {
    e = hipFuncSetAttribute((const void*)flash_fwd_kernel<T, KS, DT, 8, 2>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds2);
    if (e == hipSuccess) {
      if (frames) {
        AttnArgs ax = a;
        ax.nqb = nqb;
        ax.nb = B;
        const int64_t pairs = ((int64_t)B * a.Hq + 7) / 8 * 8;
        ax.ppx = (int)(pairs / 8);
        ax.o16 = ((uintptr_t)a.o % 16 == 0 && a.osb % 8 == 0 && a.osl % 8 == 0 && a.osh % 8 == 0) ? 1 : 0;
        static const int stream_ = [] { const char* v = getenv("TV_FA_STREAM"); return v ? atoi(v) : 1; }();
        const int64_t slots = (int64_t)ax.ppx * nqb;          // query blocks per XCD
        if constexpr (KS > 6) {                                // head_dim 128: the second Q set does not fit the registers
          flash_fwd_kernel<T, KS, DT, 8, 2><<<dim3((unsigned)(pairs * nqb), 1, 1), 512, lds2, st>>>(ax, NoSeqs{});
        } else if (stream_ && a.Lk > 32 * KT && slots > tv_cu_count() / 8) {
          // one resident work-group per CU streams its share of the query blocks
          static const int ones_ = [] { const char* v = getenv("TV_FA_ONES"); return v ? atoi(v) : 1; }();
          static const int trim_ = [] { const char* v = getenv("TV_FA_TRIM"); return v ? atoi(v) : 1; }();
          ax.notrim = !trim_;
          const dim3 grid_s((unsigned)(8 * (tv_cu_count() / 8)), 1, 1);
          const int variant = g_fa_variant.load(std::memory_order_relaxed);
          if ((variant == 0 || variant == 4) && std::is_same<T, bf16_t>::value && KS == 5 && DT == 3 && KT == 3 && ones_ && trim_ &&
              a.D % 8 == 0 && a.D < 32 * DT && a.Lk > 2 * 32 * KT) {
            // the generated tile loop (attention_vit.hpp): one wave per SIMD, 64 query rows a wave
            ax.notrim = 0;
            e = hipFuncSetAttribute((const void*)flash_fwd_vit_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e == hipSuccess) flash_fwd_vit_kernel<<<grid_s, 256, lds, st>>>(ax);
          } else if (ones_ && variant != 3 && a.D % 8 == 0 && a.D < 32 * DT) {
            e = hipFuncSetAttribute((const void*)flash_fwd_stream_kernel<T, KS, DT, KT, true>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e == hipSuccess) flash_fwd_stream_kernel<T, KS, DT, KT, true><<<grid_s, 512, lds, st>>>(ax);
          } else {
            e = hipFuncSetAttribute((const void*)flash_fwd_stream_kernel<T, KS, DT, KT, false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e == hipSuccess) flash_fwd_stream_kernel<T, KS, DT, KT, false><<<grid_s, 512, lds, st>>>(ax);
          }
        } else {
          flash_fwd_kernel<T, KS, DT, 8, 2><<<dim3((unsigned)(pairs * nqb), 1, 1), 512, lds2, st>>>(ax, NoSeqs{});
        }
      } else {
        flash_fwd_kernel<T, KS, DT, 8, 2><<<dim3((unsigned)(nqb * all)), 512, lds2, st>>>(a, NoSeqs{});
      }
    }
  }
  if (e != hipSuccess) {
    tv_set_error("flash_attn: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  TV_LAUNCH_CHECK();
}

// windowed form: bf16 (64 keys by one wave take 3 of the estimate's units, the rest of a block 13).  Blocks of 256 rows, or of 128 with two waves a row: if no sequence is longer, while those are one round, and for more where the sequences start
// from nothing and the estimate of both grids says so (one prompt, 16 heads, window 1 024: 1 200 rows 54 | 37 us, 2 560: 65 | 54, 3 200: 64 | 75; four, 3 000 together:
// 61 | 45; 32 x 100 rows behind 1 000 keys 116 | 81; but eight of 425, 16 heads 28 | 39, sixteen of 162, window 256 19 | 27).
template <int KS, int DT>
int launch_fa_win(const AttnArgs& a, const AttnSeqs& sq, int nseq, hipStream_t st) {
  constexpr int KT = 2, lds2 = fa_lds(KT);
  int most = 0;
  int64_t blocks = 0, blocks128 = 0;
  bool triangle = true;
  for (int s = 0; s < nseq; ++s) {
    most = sq.len_q[s] > most ? sq.len_q[s] : most;
    blocks += (sq.len_q[s] + 255) / 256;
    blocks128 += (sq.len_q[s] + 127) / 128;
    triangle = triangle && sq.len_k[s] - sq.len_q[s] <= sq.len_q[s] / 4;
  }
  const int64_t cus = tv_cu_count();
  bool two = most <= 128 || blocks128 * a.Hq <= cus;
  if (!two && triangle && blocks * a.Hq * 6 <= cus * (nseq < 3 ? 3 + nseq : 6)) {
    Dealt of128;
    int64_t longest = 0;
    for (int s = 0; s < nseq; ++s) {
      const int64_t start = sq.len_k[s] - sq.len_q[s];
      const auto steps = [&](int64_t q, int rows, int tile) {                     // tiles of keys that block q of the sequence visits
        const int64_t hi = std::min<int64_t>(sq.len_k[s], (q + 1) * rows + start), lo = std::max<int64_t>(0, q * rows + start - a.window + 1) / tile;
        return (hi + tile - 1) / tile - lo + std::min((std::min<int64_t>(a.keep, hi) + tile - 1) / tile, lo);
      };
      for (int64_t q = (sq.len_q[s] + 127) / 128; q-- > 0;) of128.add(10 + 4 * steps(q, 128, 128), a.Hq);
      for (int64_t q = (sq.len_q[s] + 255) / 256; q-- > 0;) longest = std::max(longest, 13 + 3 * steps(q, 256, 64));
    }
    two = dealt_out_pays(of128, longest, KS > 6);
  }
  const void* f = two ? (const void*)flash_fwd_kernel<bf16_t, KS, DT, 8, 2, true, 2> : (const void*)flash_fwd_kernel<bf16_t, KS, DT, 8, KT, true>;
  const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds2);
  if (e != hipSuccess) {
    tv_set_error("flash_attn: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  const dim3 grid((unsigned)((two ? blocks128 : blocks) * a.Hq));
  if (two) flash_fwd_kernel<bf16_t, KS, DT, 8, 2, true, 2><<<grid, 512, lds2, st>>>(a, sq);
  else flash_fwd_kernel<bf16_t, KS, DT, 8, KT, true><<<grid, 512, lds2, st>>>(a, sq);
  TV_LAUNCH_CHECK();
}

int launch_win(const AttnArgs& a, const AttnSeqs& sq, int nseq, hipStream_t st) {
  const int D = a.D > a.Dv ? a.D : a.Dv;
  if (D <= 64) return launch_fa_win<4, 2>(a, sq, nseq, st);
  if (D <= 96) return launch_fa_win<6, 3>(a, sq, nseq, st);
  return launch_fa_win<8, 4>(a, sq, nseq, st);                 // (<= 128: caller)
}

template <typename T>
int launch_fa(const AttnArgs& a, int B, hipStream_t st) {
  // One grid dimension takes fewer than 2^32 work-items: a batch with more query blocks than that goes in slices
  const int64_t blocks = (int64_t)((a.Lq + 255) / 256) * a.Hq;                        // of a batch entry, 512 work-items each
  const int64_t most = blocks < (1 << 22) ? ((1 << 23) - 64) / blocks : 1;           // (pairs are padded to a multiple of 8 in one form)
  if (B > most) {
    for (int64_t b = 0; b < B; b += most) {
      AttnArgs s = a;
      s.q = (const T*)a.q + b * a.qsb; s.k = (const T*)a.k + b * a.ksb; s.v = (const T*)a.v + b * a.vsb; s.o = (T*)a.o + b * a.osb;
      if (a.lse) s.lse = a.lse + b * a.Hq * a.Lq;
      s.nb = (int)(B - b < most ? B - b : most);
      const int rc = launch_fa<T>(s, s.nb, st);
      if (rc != TV_OK) return rc;
    }
    return TV_OK;
  }
  const int D = a.D > a.Dv ? a.D : a.Dv;
  if (D <= 64) return launch_fa_d<T, 4, 2>(a, B, st);
  if (D <= 80) return launch_fa_d<T, 5, 3>(a, B, st);
  if (D <= 96) return launch_fa_d<T, 6, 3>(a, B, st);
  if (D <= 128) return launch_fa_d<T, 8, 4>(a, B, st);
  TV_UNSUPPORTED("flash_attn: headdim %d > 128", D);
}

}  // namespace

#ifdef TV_FA_STAMP
extern "C" int tv_fa_debug_stamps(unsigned long long* out) {
  return (int)hipMemcpyFromSymbol(out, HIP_SYMBOL(g_fa_stamps), sizeof(g_fa_stamps));
}
#endif

extern "C" int tv_flash_attn_two_waves(int seqlen_q, int seqlen_k, int64_t pairs, int headdim, int causal) {
  return two_waves_a_row(seqlen_q, seqlen_k, pairs, causal != 0, headdim > 96);
}

extern "C" void tv_flash_attn_set_variant(int variant) { g_fa_variant.store(variant, std::memory_order_relaxed); }

static int flash_fwd(const void* q, const void* k, const void* v, void* o, void* lse, const float* sink, int v_dim,
                                 int batch, int seqlen_q, int seqlen_k, int nheads_q,
                                 int nheads_kv, int headdim, int64_t q_stride_b,
                                 int64_t q_stride_l, int64_t q_stride_h, int64_t k_stride_b,
                                 int64_t k_stride_l, int64_t k_stride_h, int64_t v_stride_b,
                                 int64_t v_stride_l, int64_t v_stride_h, int64_t o_stride_b,
                                 int64_t o_stride_l, int64_t o_stride_h, float softmax_scale,
                                 int causal, int dtype, void* stream) {
  TV_CHECK_ARG((seqlen_q == 0 || (q && o)) && (seqlen_q == 0 || seqlen_k == 0 || (k && v)), "flash_attn: null pointer");
  TV_CHECK_ARG(batch > 0 && seqlen_q >= 0 && seqlen_k >= 0 && nheads_q > 0 && nheads_kv > 0 &&
                   nheads_q % nheads_kv == 0 && headdim > 0 && v_dim > 0 && softmax_scale > 0.f,
               "flash_attn: bad sizes (or non-positive softmax scale)");
  if (dtype != TV_BF16 && dtype != TV_F16) TV_UNSUPPORTED("flash_attn: dtype must be bf16/f16");
  if (headdim % 8 || v_dim % 8) TV_UNSUPPORTED("flash_attn: headdim %d / %d not a multiple of 8", headdim, v_dim);
  if ((sink || v_dim != headdim) && !causal) TV_UNSUPPORTED("flash_attn: sinks and value dims of their own are causal forms");
  const int64_t strides[] = {q_stride_b, q_stride_l, q_stride_h, k_stride_b, k_stride_l,
                             k_stride_h, v_stride_b, v_stride_l, v_stride_h};
  for (int64_t s : strides)
    if (s % 8) TV_UNSUPPORTED("flash_attn: q/k/v strides must be multiples of 8 elements");
  if (o_stride_b % 4 || o_stride_l % 4 || o_stride_h % 4 || ((uintptr_t)o & 7))
    TV_UNSUPPORTED("flash_attn: o strides must be multiples of 4 elements");
  if (((uintptr_t)q & 15) || ((uintptr_t)k & 15) || ((uintptr_t)v & 15))
    TV_UNSUPPORTED("flash_attn: q/k/v must be 16-byte aligned");
  // the K/V copies address a 64-key tile with 32-bit byte offsets from its first key
  if (128 * k_stride_l * 2 >= (1ll << 31) || 128 * v_stride_l * 2 >= (1ll << 31))
    TV_UNSUPPORTED("flash_attn: k/v row stride too large");
  if (seqlen_q == 0) return TV_OK;
  AttnArgs a;
  a.q = q; a.k = k; a.v = v; a.o = o; a.lse = (float*)lse;
  a.Lq = seqlen_q; a.Lk = seqlen_k; a.Hq = nheads_q; a.Hkv = nheads_kv; a.D = headdim;
  a.qsb = q_stride_b; a.qsl = q_stride_l; a.qsh = q_stride_h;
  a.ksb = k_stride_b; a.ksl = k_stride_l; a.ksh = k_stride_h;
  a.vsb = v_stride_b; a.vsl = v_stride_l; a.vsh = v_stride_h;
  a.osb = o_stride_b; a.osl = o_stride_l; a.osh = o_stride_h;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  a.causal = causal;
  a.nqb = 0;
  a.nb = batch;
  a.Dv = v_dim;
  a.sink = sink;
  a.window = a.keep = 0; a.gate = nullptr; a.gsl = a.gsh = 0;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TV_BF16) return launch_fa<bf16_t>(a, batch, st);
  return launch_fa<f16_t>(a, batch, st);
}

extern "C" int tv_flash_attn_fwd(const void* q, const void* k, const void* v, void* o, void* lse,
                                 int batch, int seqlen_q, int seqlen_k, int nheads_q,
                                 int nheads_kv, int headdim, int64_t q_stride_b,
                                 int64_t q_stride_l, int64_t q_stride_h, int64_t k_stride_b,
                                 int64_t k_stride_l, int64_t k_stride_h, int64_t v_stride_b,
                                 int64_t v_stride_l, int64_t v_stride_h, int64_t o_stride_b,
                                 int64_t o_stride_l, int64_t o_stride_h, float softmax_scale,
                                 int causal, int dtype, void* stream) {
  return flash_fwd(q, k, v, o, lse, nullptr, headdim, batch, seqlen_q, seqlen_k, nheads_q, nheads_kv, headdim, q_stride_b, q_stride_l,
                   q_stride_h, k_stride_b, k_stride_l, k_stride_h, v_stride_b, v_stride_l, v_stride_h, o_stride_b, o_stride_l, o_stride_h,
                   softmax_scale, causal, dtype, stream);
}

// Causal attention with a sink logit per q-head (exp(sink) joins the denominator, unscaled) and a value dim of its own.
extern "C" int tv_flash_attn_sink_fwd(const void* q, const void* k, const void* v, void* o, const float* sink, int v_dim,
                                 int batch, int seqlen_q, int seqlen_k, int nheads_q,
                                 int nheads_kv, int headdim, int64_t q_stride_b,
                                 int64_t q_stride_l, int64_t q_stride_h, int64_t k_stride_b,
                                 int64_t k_stride_l, int64_t k_stride_h, int64_t v_stride_b,
                                 int64_t v_stride_l, int64_t v_stride_h, int64_t o_stride_b,
                                 int64_t o_stride_l, int64_t o_stride_h, float softmax_scale,
                                 int dtype, void* stream) {
  return flash_fwd(q, k, v, o, nullptr, sink, v_dim, batch, seqlen_q, seqlen_k, nheads_q, nheads_kv, headdim, q_stride_b, q_stride_l,
                   q_stride_h, k_stride_b, k_stride_l, k_stride_h, v_stride_b, v_stride_l, v_stride_h, o_stride_b, o_stride_l, o_stride_h,
                   softmax_scale, 1, dtype, stream);
}

// Causal attention of one sequence with a sliding window and kept first keys, a value dim of its own and an optional output gate
// (o *= sigmoid(gate)); bf16.
extern "C" int tv_flash_attn_window_fwd(const void* q, const void* k, const void* v, void* o, const void* gate, int window,
                                        int keep_first, int v_dim, int seqlen_q, int seqlen_k, int nheads_q, int nheads_kv, int headdim,
                                        int64_t q_stride_l, int64_t q_stride_h, int64_t k_stride_l, int64_t k_stride_h,
                                        int64_t v_stride_l, int64_t v_stride_h, int64_t o_stride_l, int64_t o_stride_h,
                                        int64_t gate_stride_l, int64_t gate_stride_h, float softmax_scale, int dtype, void* stream) {
  const int zero = 0;
  return tv_flash_attn_window_packed_fwd(q, k, v, o, gate, window, keep_first, v_dim, 1, &zero, &seqlen_q, &seqlen_k, &zero, nheads_q, nheads_kv, headdim,
                                         q_stride_l, q_stride_h, 0, k_stride_l, k_stride_h, 0, v_stride_l, v_stride_h, o_stride_l, o_stride_h,
                                         gate_stride_l, gate_stride_h, softmax_scale, dtype, stream);
}

// The same for the sequences of a packed step: sequence s owns rows [rows[s], rows[s] + lens_q[s]) of q, o and gate and sees the first
// lens_k[s] rows of batch entry slots[s] of k and v (host arrays, read before the call returns).
extern "C" int tv_flash_attn_window_packed_fwd(const void* q, const void* k, const void* v, void* o, const void* gate, int window, int keep_first,
                                               int v_dim, int nseq, const int* rows, const int* lens_q, const int* lens_k, const int* slots,
                                               int nheads_q, int nheads_kv, int headdim, int64_t q_stride_l, int64_t q_stride_h,
                                               int64_t k_stride_b, int64_t k_stride_l, int64_t k_stride_h, int64_t v_stride_b,
                                               int64_t v_stride_l, int64_t v_stride_h, int64_t o_stride_l, int64_t o_stride_h,
                                               int64_t gate_stride_l, int64_t gate_stride_h, float softmax_scale, int dtype, void* stream) {
  TV_CHECK_ARG(nseq >= 0 && (nseq == 0 || (rows && lens_q && lens_k && slots)), "flash_attn_window: sequences");
  int64_t total = 0;
  for (int s = 0; s < nseq; ++s) {
    TV_CHECK_ARG(rows[s] >= 0 && lens_q[s] >= 0 && slots[s] >= 0 && lens_k[s] >= lens_q[s], "flash_attn_window: bad window or lengths");
    total += lens_q[s];
  }
  TV_CHECK_ARG(window > 0 && keep_first >= 0, "flash_attn_window: bad window or lengths");
  TV_CHECK_ARG(total == 0 || (q && o && k && v), "flash_attn: null pointer");
  TV_CHECK_ARG(nheads_q > 0 && nheads_kv > 0 && nheads_q % nheads_kv == 0 && headdim > 0 && v_dim > 0 && softmax_scale > 0.f,
               "flash_attn: bad sizes (or non-positive softmax scale)");
  if (dtype != TV_BF16) TV_UNSUPPORTED("flash_attn_window: dtype must be bf16");
  if (headdim % 8 || v_dim % 8) TV_UNSUPPORTED("flash_attn: headdim %d / %d not a multiple of 8", headdim, v_dim);
  if (headdim > 128 || v_dim > 128) TV_UNSUPPORTED("flash_attn_window: headdim %d / %d > 128", headdim, v_dim);
  if (gate && (gate_stride_l % 4 || gate_stride_h % 4 || ((uintptr_t)gate & 7)))
    TV_UNSUPPORTED("flash_attn_window: gate rows must be 8-byte aligned");
  const int64_t strides[] = {q_stride_l, q_stride_h, k_stride_b, k_stride_l, k_stride_h, v_stride_b, v_stride_l, v_stride_h};
  for (int64_t s : strides)
    if (s % 8) TV_UNSUPPORTED("flash_attn: q/k/v strides must be multiples of 8 elements");
  if (o_stride_l % 4 || o_stride_h % 4 || ((uintptr_t)o & 7)) TV_UNSUPPORTED("flash_attn: o strides must be multiples of 4 elements");
  if (((uintptr_t)q & 15) || ((uintptr_t)k & 15) || ((uintptr_t)v & 15)) TV_UNSUPPORTED("flash_attn: q/k/v must be 16-byte aligned");
  if (128 * k_stride_l * 2 >= (1ll << 31) || 128 * v_stride_l * 2 >= (1ll << 31)) TV_UNSUPPORTED("flash_attn: k/v row stride too large");
  if (total == 0) return TV_OK;
  AttnArgs a{};
  a.q = q; a.k = k; a.v = v; a.o = o;
  a.Hq = nheads_q; a.Hkv = nheads_kv; a.D = headdim; a.Dv = v_dim;
  a.qsl = q_stride_l; a.qsh = q_stride_h; a.ksb = k_stride_b; a.ksl = k_stride_l; a.ksh = k_stride_h;
  a.vsb = v_stride_b; a.vsl = v_stride_l; a.vsh = v_stride_h; a.osl = o_stride_l; a.osh = o_stride_h;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  a.causal = 1;
  a.window = window; a.keep = keep_first; a.gate = gate; a.gsl = gate_stride_l; a.gsh = gate_stride_h;
  // FA_SEQS sequences a launch, the longest of them first
  for (int i = 0; i < nseq;) {
    AttnSeqs sq{};
    int n = 0;
    for (; i < nseq && n < FA_SEQS; ++i) {
      if (lens_q[i] == 0) continue;
      int j = n++;
      for (; j > 0 && sq.len_k[j - 1] < lens_k[i]; --j) {
        sq.row[j] = sq.row[j - 1]; sq.len_q[j] = sq.len_q[j - 1]; sq.len_k[j] = sq.len_k[j - 1]; sq.slot[j] = sq.slot[j - 1];
      }
      sq.row[j] = rows[i]; sq.len_q[j] = lens_q[i]; sq.len_k[j] = lens_k[i]; sq.slot[j] = slots[i];
    }
    const int rc = n ? launch_win(a, sq, n, (hipStream_t)stream) : TV_OK;
    if (rc != TV_OK) return rc;
  }
  return TV_OK;
}
