// Linear attention with one constant decay per head (see lightning.hip) on the matrix cores: bf16 prompts, head sizes up to 128.
//
// Chunks of 64 tokens.  Inside a chunk, with w_n = decay^n (fp32 throughout the weights, the state and the sums):
//     o_i = w_(i+1) S^T q_i + sum_(j <= i) w_(i-j) (q_i . k_j) v_j          S: the state in front of the chunk
//     S  <- w_64 S + sum_j (w_(63-j) k_j) v_j^T
// A work-group of 8 waves marches one head of one sequence through a SEGMENT of tokens; long prompts are cut into segments that
// run concurrently: a first launch computes the state behind the first segment and what each later one adds to a zero state (and
// sets the sequence's state aside: the last segment overwrites it), and the second folds the segments in front of its own into
// its starting state.
//
// Products (v_mfma_f32_16x16x32_bf16), T = transposed:
//     P^T[j][i]  = K . Q^T          K rows permuted so that a lane's accumulators are the 8 consecutive j its PV fragment needs
//     O^T[e][i]  = S^T . Q^T, scaled by w_(i+1) per lane, + V^T . P^T
//     S[d][e]   += (w K)^T . V
// V^T, (w K)^T and V come out of row-major LDS tiles through transposing reads.  The operands that are not bf16 by nature —
// P, w K and the state S — are split into two bf16 terms (high + remainder): the products keep 32-bit weights and state.
#include "lightning.hpp"

namespace {

typedef __attribute__((address_space(3))) bf16x4 lm_lds4;
typedef __attribute__((address_space(3))) const bf16x8 lm_lds8;

constexpr int LM_THREADS = 512;
constexpr int LM_Q = 64;              // tokens per chunk

struct LmArgs {
  const bf16_t *q, *k, *v;
  const float* decay;
  float *state, *part;                // part, nseg > 1: [nseq][H][nseg][dk][dv] — states of segments 0 .. nseg - 2, then the state
                                      // the sequence came with
  bf16_t* o;
  const int *cu, *slot;
  int H, dk, dv, silu, nseg, seglen;
  int64_t qs, ks, vs, os;
};

__device__ __forceinline__ f32x4 mm(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ bf16x8 silu8(bf16x8 x) {
  bf16x8 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float f = (float)x[i];
    r[i] = (bf16_t)(f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * f)));
  }
  return r;
}

__device__ __forceinline__ void split8(const float (&x)[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hi[i] = (bf16_t)x[i];
    lo[i] = (bf16_t)(x[i] - (float)hi[i]);
  }
}

// rows 8 g .. 8 g + 7 of column c0 + lc of a row-major tile (row stride `rs` bytes): the k-major operand fragment of a lane
__device__ __forceinline__ bf16x8 tr_frag(unsigned base, unsigned rs, int lane) {
  const int n = lane & 15, g = lane >> 4;
  const unsigned p = base + (unsigned)(8 * g + (n >> 2)) * rs + 8u * (n & 3);
  const bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lm_lds4*)(size_t)p);
  const bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lm_lds4*)(size_t)(p + 4 * rs));
  return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

template <int DK, int DV>
struct LmLds {
  static constexpr unsigned RK = DK * 2 + 32, RV = DV * 2 + 32;      // row strides: 32 bytes of padding turn the banks
  static constexpr unsigned Q = 0, K = Q + LM_Q * RK, V = K + LM_Q * RK, SH = V + LM_Q * RV, SL = SH + DV * RK, W = SL + DV * RK,
                            BYTES = W + 65 * 4 + 12;
};

// STATE: only what the segment adds to a zero state
template <int DK, int DV, bool STATE>
__global__ __launch_bounds__(LM_THREADS) void lightning_mfma_kernel(LmArgs a) {
  typedef LmLds<DK, DV> L;
  constexpr int DT = DK / 16, NT = DV / 16;          // tiles of the state
  constexpr int GR = 8 / DT;                         // waves that share a key tile of the state
  constexpr int SN = NT / GR;                        // value tiles of the state per wave
  constexpr int ON = NT / 2;                         // value tiles of the output per wave
  constexpr int QP = LM_Q * DK / 8 / LM_THREADS, VP = LM_Q * DV / 8 / LM_THREADS;      // 16-byte pieces per thread
  extern __shared__ __attribute__((aligned(16))) unsigned char lm_smem[];
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lm_smem;
  float* sw = (float*)(lm_smem + L::W);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, kq = lane >> 4;
  const int seg = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int64_t row0 = a.cu[b];
  const int n = a.cu[b + 1] - (int)row0;
  const int t_begin = seg * a.seglen, t_end = min(n, t_begin + a.seglen);
  if (t_begin >= n || (STATE && t_end >= n)) return;          // (the last segment's sum is never asked for)
  const float dec = a.decay[h];
  const float l2 = log2f(dec);                              // -inf at decay 0: the table below does not multiply it by 0
  if (tid <= 64) sw[tid] = tid == 0 ? 1.f : __builtin_amdgcn_exp2f((float)tid * l2);

  // ---- starting state of this wave's tiles: key tile wave % DT, value tiles SN (wave / DT) ..
  const int dt = wave % DT, nt0 = SN * (wave / DT);
  float* Sg = a.state + ((int64_t)a.slot[b] * a.H + h) * a.dk * a.dv;
  const int64_t blk = (int64_t)a.dk * a.dv;
  float* pp = a.part + ((int64_t)b * a.H + h) * a.nseg * blk;
  f32x4 S[SN];
  auto at = [&](int s, int r) __attribute__((always_inline)) { return (int64_t)(16 * dt + 4 * kq + r) * a.dv + 16 * (nt0 + s) + lc; };
  auto inside = [&](int s, int r) __attribute__((always_inline)) { return 16 * dt + 4 * kq + r < a.dk && 16 * (nt0 + s) + lc < a.dv; };
  // first segment: the sequence's state (of a longer sequence: the copy the first launch has set aside); later ones: the state
  // behind the first segment and the sums of those in between
  const float* from = seg == 0 ? (!STATE && n > a.seglen ? pp + (a.nseg - 1) * blk : Sg) : (STATE ? nullptr : pp);
#pragma unroll
  for (int s = 0; s < SN; ++s)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      S[s][r] = from && inside(s, r) ? from[at(s, r)] : 0.f;
      if (STATE && seg == 0 && inside(s, r)) pp[(a.nseg - 1) * blk + at(s, r)] = S[s][r];
    }
  if (!STATE && seg > 1) {
    const float dseg = dec > 0.f ? __builtin_amdgcn_exp2f((float)a.seglen * l2) : 0.f;
    for (int j = 1; j < seg; ++j) {
      const float* pj = pp + j * blk;
#pragma unroll
      for (int s = 0; s < SN; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[s][r] = fmaf(dseg, S[s][r], inside(s, r) ? pj[at(s, r)] : 0.f);
    }
  }

  // ---- copies: global -> registers a chunk ahead, activation and zero fill on the way into LDS
  bf16x8 qr[QP], kr[QP], vr[VP];
  auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < QP; ++j) {
      const int i = tid + LM_THREADS * j, r = i / (DK / 8), c = 8 * (i % (DK / 8));
      const bool ok = t0 + r < t_end && c < a.dk;
      const int64_t row = row0 + t0 + r;
      const bf16x8 z = {};
      if (!STATE) qr[j] = ok ? *(const bf16x8*)(a.q + row * a.qs + (int64_t)h * a.dk + c) : z;
      kr[j] = ok ? *(const bf16x8*)(a.k + row * a.ks + (int64_t)h * a.dk + c) : z;
    }
#pragma unroll
    for (int j = 0; j < VP; ++j) {
      const int i = tid + LM_THREADS * j, r = i / (DV / 8), c = 8 * (i % (DV / 8));
      const bf16x8 z = {};
      vr[j] = t0 + r < t_end && c < a.dv ? *(const bf16x8*)(a.v + (row0 + t0 + r) * a.vs + (int64_t)h * a.dv + c) : z;
    }
  };
  auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < QP; ++j) {
      const int i = tid + LM_THREADS * j, r = i / (DK / 8), c = i % (DK / 8);
      if (!STATE) *(bf16x8*)(lm_smem + L::Q + r * L::RK + 16 * c) = a.silu ? silu8(qr[j]) : qr[j];
      *(bf16x8*)(lm_smem + L::K + r * L::RK + 16 * c) = a.silu ? silu8(kr[j]) : kr[j];
    }
#pragma unroll
    for (int j = 0; j < VP; ++j) {
      const int i = tid + LM_THREADS * j, r = i / (DV / 8), c = i % (DV / 8);
      *(bf16x8*)(lm_smem + L::V + r * L::RV + 16 * c) = a.silu ? silu8(vr[j]) : vr[j];
    }
  };
  fetch(t_begin);
  __syncthreads();                                            // the weight table

  const int w4 = wave & 3, oh = ON * (wave >> 2);             // this wave's token tile and value tiles of the output
  const int ti = 16 * w4 + lc;                                // its lane's token in the chunk
  float pw[2][8], kw[2][8];                                   // weights of P^T and of the keys in the state update
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = 32 * p + 8 * kq + i;
      pw[p][i] = j <= ti ? sw[ti - j] : 0.f;
      kw[p][i] = sw[63 - j];
    }
  const float wi = sw[ti + 1];

  for (int t0 = t_begin; t0 < t_end; t0 += LM_Q) {
    const int tt = min(LM_Q, t_end - t0);
    put();
    if (!STATE) {
#pragma unroll
      for (int s = 0; s < SN; ++s) {                          // S^T rows e, 4 consecutive d: two bf16 terms
        bf16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          hi[r] = (bf16_t)S[s][r];
          lo[r] = (bf16_t)(S[s][r] - (float)hi[r]);
        }
        const unsigned off = (16 * (nt0 + s) + lc) * L::RK + 2 * (16 * dt + 4 * kq);
        *(bf16x4*)(lm_smem + L::SH + off) = hi;
        *(bf16x4*)(lm_smem + L::SL + off) = lo;
      }
    }
    if (tt < LM_Q) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int j = 32 * p + 8 * kq + i;
          kw[p][i] = j < tt ? sw[tt - 1 - j] : 0.f;
        }
    }
    __syncthreads();
    if (t0 + LM_Q < t_end) fetch(t0 + LM_Q);

    if (!STATE) {
      bf16x8 qf[DK / 32];
#pragma unroll
      for (int ks = 0; ks < DK / 32; ++ks) qf[ks] = *(lm_lds8*)(size_t)(lds + L::Q + ti * L::RK + 64 * ks + 16 * kq);
      f32x4 O[ON];
#pragma unroll
      for (int e = 0; e < ON; ++e) {
        O[e] = f32x4{0.f, 0.f, 0.f, 0.f};
        const unsigned sr = (16 * (oh + e) + lc) * L::RK + 16 * kq;
#pragma unroll
        for (int ks = 0; ks < DK / 32; ++ks) {
          O[e] = mm(*(lm_lds8*)(size_t)(lds + L::SH + sr + 64 * ks), qf[ks], O[e]);
          O[e] = mm(*(lm_lds8*)(size_t)(lds + L::SL + sr + 64 * ks), qf[ks], O[e]);
        }
        O[e] *= wi;
      }
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (p == 1 && w4 < 2) break;                          // (keys behind every token of this wave)
        float pv[8];
#pragma unroll
        for (int G = 0; G < 2; ++G) {
          f32x4 c = {0.f, 0.f, 0.f, 0.f};
          const unsigned kr_ = lds + L::K + (32 * p + 8 * (lc >> 2) + 4 * G + (lc & 3)) * L::RK + 16 * kq;
#pragma unroll
          for (int ks = 0; ks < DK / 32; ++ks) c = mm(*(lm_lds8*)(size_t)(kr_ + 64 * ks), qf[ks], c);
#pragma unroll
          for (int r = 0; r < 4; ++r) pv[4 * G + r] = c[r] * pw[p][4 * G + r];
        }
        bf16x8 hi, lo;
        split8(pv, hi, lo);
#pragma unroll
        for (int e = 0; e < ON; ++e) {
          const bf16x8 vf = tr_frag(lds + L::V + 32 * p * L::RV + 32 * (oh + e), L::RV, lane);
          O[e] = mm(vf, hi, O[e]);
          O[e] = mm(vf, lo, O[e]);
        }
      }
      if (ti < tt) {
        bf16_t* op = a.o + (row0 + t0 + ti) * a.os + (int64_t)h * a.dv + 4 * kq;
#pragma unroll
        for (int e = 0; e < ON; ++e)
          if (16 * (oh + e) + 4 * kq < a.dv) {
            bf16x4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = (bf16_t)O[e][r];
            *(bf16x4*)(op + 16 * (oh + e)) = y;
          }
      }
    }
    const float wt = sw[tt];
#pragma unroll
    for (int s = 0; s < SN; ++s) S[s] *= wt;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const bf16x8 kf = tr_frag(lds + L::K + 32 * p * L::RK + 32 * dt, L::RK, lane);
      float kv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) kv[i] = (float)kf[i] * kw[p][i];
      bf16x8 hi, lo;
      split8(kv, hi, lo);
#pragma unroll
      for (int s = 0; s < SN; ++s) {
        const bf16x8 vf = tr_frag(lds + L::V + 32 * p * L::RV + 32 * (nt0 + s), L::RV, lane);
        S[s] = mm(hi, vf, S[s]);
        S[s] = mm(lo, vf, S[s]);
      }
    }
    __syncthreads();                                          // the tiles are written again
  }
  float* out = STATE ? pp + seg * blk : Sg;
  if (STATE || t_end == n) {
#pragma unroll
    for (int s = 0; s < SN; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (inside(s, r)) out[at(s, r)] = S[s][r];
  }
}

template <int DK, int DV>
int launch_dims(const LmArgs& a, int nseq, hipStream_t st) {
  constexpr int lds = LmLds<DK, DV>::BYTES;
  hipError_t e = hipFuncSetAttribute((const void*)lightning_mfma_kernel<DK, DV, false>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess) e = hipFuncSetAttribute((const void*)lightning_mfma_kernel<DK, DV, true>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) {
    tv_set_error("lightning: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  if (a.nseg > 1)
    lightning_mfma_kernel<DK, DV, true><<<dim3((unsigned)(a.nseg - 1), (unsigned)a.H, (unsigned)nseq), LM_THREADS, lds, st>>>(a);
  lightning_mfma_kernel<DK, DV, false><<<dim3((unsigned)a.nseg, (unsigned)a.H, (unsigned)nseq), LM_THREADS, lds, st>>>(a);
  TV_LAUNCH_CHECK();
}

}  // namespace

// segments per sequence: one work-group per compute unit, at least 4 chunks each
void tv_lightning_segments(int nseq, int nheads, int max_len, int* nseg, int* seglen) {
  const int chunks = (max_len + LM_Q - 1) / LM_Q;
  int want = tv_cu_count() / (nseq * nheads > 0 ? nseq * nheads : 1);
  if (want > (chunks + 3) / 4) want = (chunks + 3) / 4;
  if (want < 1) want = 1;
  const int per = (chunks + want - 1) / want;
  *seglen = per * LM_Q;
  *nseg = (chunks + per - 1) / per;
  if (*nseg < 1) *nseg = 1;
}

bool tv_lightning_mfma_takes(const void* q, const void* k, const void* v, const void* o, int dk, int dv, int64_t qs, int64_t ks, int64_t vs,
                             int64_t os, int dtype) {
  auto ok = [](const void* p, int64_t s) { return ((uintptr_t)p & 15) == 0 && s % 8 == 0; };
  return dtype == TV_BF16 && dk % 8 == 0 && dv % 8 == 0 && dk <= 128 && dv <= 128 && ok(q, qs) && ok(k, ks) && ok(v, vs) &&
         ((uintptr_t)o & 7) == 0 && os % 4 == 0;
}

int tv_lightning_mfma_launch(const void* q, const void* k, const void* v, const float* decay, float* state, void* o, const int* cu,
                             const int* slot, int nseq, int H, int dk, int dv, int64_t qs, int64_t ks, int64_t vs, int64_t os, int silu,
                             int nseg, int seglen, float* part, hipStream_t st) {
  LmArgs a{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, decay, state, part, (bf16_t*)o, cu, slot, H, dk, dv, silu, nseg, seglen,
           qs, ks, vs, os};
  if (dk <= 64) return dv <= 64 ? launch_dims<64, 64>(a, nseq, st) : launch_dims<64, 128>(a, nseq, st);
  return dv <= 64 ? launch_dims<128, 64>(a, nseq, st) : launch_dims<128, 128>(a, nseq, st);
}
