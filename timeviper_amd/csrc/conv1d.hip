// S2: causal depthwise conv1d (+bias +SiLU), channels-last.
// Each lane owns 16 bytes of channels of a strip of 8 consecutive tokens: all its rows in flight at once, fully coalesced, then a K-row
// register window slides down them.  The K-1 rows in front of a strip are read again, from a cache.
// Long sequences are bound by HBM (5.3 TB/s of x once in and once out), short ones by the one round trip to memory and the weights' loads in
// front of it.  8 tokens, because a longer strip's rows come in several round trips; 12 288 channels, bf16, all with C.B^T, us for strips
// of 8 | 16 | 32 | 64: 203 tokens 6.3 | 7.2 | 11.2 | 19.3, 1 501: 17 | 16 | 17 | 23, 49 999: 467 | 472 | 486 | 505 (of 4: 508).  With 64, weights
// loaded two bytes at a time and B / C in a launch of their own it was 33, 35 and 534 us.
// Reference semantics: modeling_nano.py:619-624 / :705 (zero left pad).
#include "ssd_common.hpp"

namespace {

constexpr int CONV_THREADS = 256;
constexpr int CONV_TL = 8;       // tokens a strip

// A lane's V channels: V K weights = K 16-byte vectors, where w and bias are aligned (wide); else one by one
template <typename T, int K>
struct ConvTaps {
  enum { V = Vec16<T>::N };
  float wk[K][V], bs[V];
  __device__ __forceinline__ void load(const T* __restrict__ w, const T* __restrict__ bias, int c0, int wide) {
    typedef typename Vec16<T>::type vec_t;
    if (wide) {
      vec_t wv[K], bv = {};
#pragma unroll
      for (int j = 0; j < K; ++j) wv[j] = *(const vec_t*)(w + (int64_t)c0 * K + j * V);
      if (bias) bv = *(const vec_t*)(bias + c0);
#pragma unroll
      for (int i = 0; i < V; ++i) {
#pragma unroll
        for (int j = 0; j < K; ++j) wk[j][i] = to_f32(wv[(i * K + j) / V][(i * K + j) % V]);
        bs[i] = to_f32(bv[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) {
#pragma unroll
        for (int j = 0; j < K; ++j) wk[j][i] = to_f32(w[(int64_t)(c0 + i) * K + j]);
        bs[i] = bias ? to_f32(bias[c0 + i]) : 0.f;
      }
    }
  }
};

struct ConvArgs {
  const void *x, *w, *bias, *halo;
  void *yx, *yb, *yc, *cb;       // the plain form writes yx alone
  int L, C, d_inner, G, N, silu, wide;
  int nxb, per_xcd;              // blocks a strip of tokens; strips an XCD
  int nchunks, nbc;              // blocks of the B / C part (0: its channels are in the strips)
  int64_t xsb, xsl, ysb, ysl;
};

// A block's strip and channels: each XCD has a run of strips, so that the rows in front of a strip are in its L2 (4 096 tokens x 12 288
// channels: 40.5 -> 35.5 us; no difference where a run is larger than the L2)
template <typename T>
__device__ __forceinline__ bool conv_place(const ConvArgs& a, int block, int c_end, int& c0, int& t0) {
  const int xcd = block & 7, j = block >> 3;
  c0 = (j % a.nxb * CONV_THREADS + (int)threadIdx.x) * Vec16<T>::N;
  t0 = (xcd * a.per_xcd + j / a.nxb) * CONV_TL;
  return c0 < c_end && t0 < a.L;
}

// One lane's strip of CONV_TL rows from t0 on, of a sequence of L: all its rows and the K-1 in front of it are in flight before the
// arithmetic; rows past the end repeat the last one and are left out of it.  FAST: SiLU with the reciprocal instruction (the mixer's convolution).
template <typename T, int K, bool FAST>
__device__ __forceinline__ void conv_strip(const ConvArgs& a, int c0, int t0, int b, T* __restrict__ yb, int64_t ysl) {
  constexpr int V = Vec16<T>::N;
  typedef typename Vec16<T>::type vec_t;
  const T* xb = (const T*)a.x + (int64_t)b * a.xsb + c0;
  const T* hb = a.halo ? (const T*)a.halo + (int64_t)b * (K - 1) * a.C + c0 : nullptr;
  vec_t v[K - 1 + CONV_TL];
#pragma unroll
  for (int j = 0; j < K - 1; ++j) {
    const int t = t0 - (K - 1) + j;
    v[j] = vec_t{};
    if (t >= 0) v[j] = *(const vec_t*)(xb + (int64_t)t * a.xsl);
    else if (hb) v[j] = *(const vec_t*)(hb + (int64_t)(t + K - 1) * a.C);
  }
#pragma unroll
  for (int u = 0; u < CONV_TL; ++u) v[K - 1 + u] = *(const vec_t*)(xb + (int64_t)min(t0 + u, a.L - 1) * a.xsl);
  ConvTaps<T, K> tp;
  tp.load((const T*)a.w, (const T*)a.bias, c0, a.wide);
  float win[K][V];               // win[j] holds row t-(K-1)+j
#pragma unroll
  for (int j = 0; j < K - 1; ++j)
#pragma unroll
    for (int i = 0; i < V; ++i) win[j][i] = to_f32(v[j][i]);
#pragma unroll
  for (int u = 0; u < CONV_TL; ++u) {
    if (t0 + u >= a.L) break;                      // (the same for all lanes; one row of 4 096 channels 5.3 us with all eight computed)
    vec_t ov;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      win[K - 1][i] = to_f32(v[K - 1 + u][i]);
      float acc = tp.bs[i];
#pragma unroll
      for (int j = 0; j < K; ++j) acc = fmaf(tp.wk[j][i], win[j][i], acc);
      if (a.silu) acc = FAST ? acc * __builtin_amdgcn_rcpf(1.f + __expf(-acc)) : silu_f(acc);
      ov[i] = from_f32<T>(acc);
#pragma unroll
      for (int j = 0; j < K - 1; ++j) win[j][i] = win[j + 1][i];
    }
    *(vec_t*)(yb + (int64_t)(t0 + u) * ysl) = ov;
  }
}

template <typename T, int K>
__global__ __launch_bounds__(CONV_THREADS) void conv1d_fwd_kernel(ConvArgs a) {
  int c0, t0;
  if (!conv_place<T>(a, blockIdx.x, a.C, c0, t0)) return;
  conv_strip<T, K, false>(a, c0, t0, blockIdx.y, (T*)a.yx + (int64_t)blockIdx.y * a.ysb + c0, a.ysl);
}

// Mamba-2 xBC variant: the three channel segments go to three destinations; B and C are
// written group-major (B,G,L,N) so that one group's consecutive tokens are contiguous.
template <typename T, int K>
__device__ __forceinline__ void conv_xbc_block(const ConvArgs& a, int block, int b, int c_end) {
  int c0, t0;
  if (!conv_place<T>(a, block, c_end, c0, t0)) return;
  // destination of this lane's 16 bytes: row pointer at t=0 and row stride
  T* yb;
  int64_t ysl;
  const int gn = a.G * a.N;
  if (c0 < a.d_inner) {
    yb = (T*)a.yx + (int64_t)b * a.L * a.d_inner + c0;
    ysl = a.d_inner;
  } else {
    const bool isB = c0 < a.d_inner + gn;
    const int cc = c0 - a.d_inner - (isB ? 0 : gn);
    const int g = cc / a.N, n = cc - g * a.N;
    yb = (T*)(isB ? a.yb : a.yc) + ((int64_t)b * a.G + g) * a.L * a.N + n;
    ysl = a.N;
  }
  conv_strip<T, K, true>(a, c0, t0, b, yb, ysl);
}
template <typename T, int K>
__global__ __launch_bounds__(CONV_THREADS) void conv1d_xbc_kernel(ConvArgs a) {
  conv_xbc_block<T, K>(a, blockIdx.x, blockIdx.y, a.C);
}


// ------------------------------------------------------------------ B / C channels + causal C.B^T of a chunk
// The B and C channels of ONE (64-token chunk, group): convolution + SiLU exactly as conv1d_xbc_kernel
// (same fp32 operations in the same order), group-major stores — and, while the chunk's 64 x 128 B and C tiles are
// still on the chip (LDS), the causal part of C.B^T in the fragment order the scan kernel's mask waves read
// (ssd_slice.hip: 6 fragments of 512 bf16 per (chunk, group); fragment (ti, sp), lane (lc, kq) holds
// CB[16 ti + lc][32 sp + 8 kq + 0..7]).  A pre-pass of the scan that reads B and C back from
// memory costs 0.8 GB and ~100 us per layer at 164 k tokens.
// 256 threads: thread = (strip of 8 tokens, 16 bytes of the group's 256 B / C channels).
constexpr int CBQ = 64, CBN = 128, CB_FRAGS = 6;
template <int K>
__device__ __forceinline__ void conv_bc_cb_block(const ConvArgs& a, bf16_t (*tile)[CBQ * CBN], int c, int g, int b) {
  using namespace ssdk;                                    // tile: [B | C][token][n], 16-byte chunk ^ (token & 15)
  const int tid = threadIdx.x, L = a.L, C = a.C, silu = a.silu;
  const int64_t xsl = a.xsl;
  const int strip = tid >> 5, l32 = tid & 31;
  const int isC = l32 >> 4, nch = l32 & 15;                // 16-byte chunk of the group's 128 states
  const int c0 = a.d_inner + (isC ? a.G * CBN : 0) + g * CBN + nch * 8;
  const int t0 = c * CBQ + strip * 8;
  const bf16_t* xb = (const bf16_t*)a.x + (int64_t)b * a.xsb + c0;
  const bf16_t* hb = a.halo ? (const bf16_t*)a.halo + (int64_t)b * (K - 1) * C + c0 : nullptr;
  bf16_t* yg = (bf16_t*)(isC ? a.yc : a.yb) + ((int64_t)b * a.G + g) * L * CBN + nch * 8;
  bf16_t* tl = tile[isC];
  // all rows of the strip (and its K-1 predecessors) in flight, then the arithmetic
  bf16x8 v[K - 1 + 8];
#pragma unroll
  for (int j = 0; j < K - 1 + 8; ++j) {
    const int t = t0 - (K - 1) + j;
    v[j] = bf16x8{};
    if (t >= 0 && t < L) v[j] = *(const bf16x8*)(xb + (int64_t)t * xsl);
    else if (t < 0 && hb) v[j] = *(const bf16x8*)(hb + (int64_t)(t + K - 1) * C);
  }
  ConvTaps<bf16_t, K> tp;
  tp.load((const bf16_t*)a.w, (const bf16_t*)a.bias, c0, a.wide);
  float win[K][8];
#pragma unroll
  for (int j = 0; j < K - 1; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) win[j][i] = to_f32(v[j][i]);
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int t = t0 + u;
    bf16x8 ov;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      win[K - 1][i] = to_f32(v[K - 1 + u][i]);
      float acc = tp.bs[i];
#pragma unroll
      for (int j = 0; j < K; ++j) acc = fmaf(tp.wk[j][i], win[j][i], acc);
      if (silu) acc *= __builtin_amdgcn_rcpf(1.f + __expf(-acc));   // x * sigmoid(x)
      ov[i] = (bf16_t)acc;
#pragma unroll
      for (int j = 0; j < K - 1; ++j) win[j][i] = win[j + 1][i];
    }
    if (t >= L) ov = bf16x8{};                    // rows past the sequence end: finite, never stored
    else *(bf16x8*)(yg + (int64_t)t * CBN) = ov;
    const int row = strip * 8 + u;
    *(bf16x8*)(tl + row * CBN + ((nch ^ (row & 15)) << 3)) = ov;
  }
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6;
  if (wave == 3) return;
  const int lc = lane & 15, kq = lane >> 4;
  // as ssd_cb_kernel: wave 0: fragments (2,0) (2,1); wave 1: (3,0) (3,1); wave 2: (0,0) (1,0)
  const int nct = wave == 2 ? 2 : 1, nsp = wave == 2 ? 1 : 2;
  const int ti0 = wave == 0 ? 2 : wave == 1 ? 3 : 0;
  auto rd = [&](const bf16_t* tlp, int row, int ks) {
    return *(const bf16x8*)(tlp + row * CBN + (((4 * ks + kq) ^ (row & 15)) << 3));
  };
  bf16x8 cf[2][4], b0[2][4], b1[2][4];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (u < nct) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) cf[u][ks] = rd(tile[1], 16 * (ti0 + u) + lc, ks);
    }
    if (u < nsp) {
      const int s_lo = 32 * u + 8 * (lc >> 2) + (lc & 3);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        b0[u][ks] = rd(tile[0], s_lo, ks);
        b1[u][ks] = rd(tile[0], s_lo + 4, ks);
      }
    }
  }
#pragma unroll
  for (int ff = 0; ff < 2; ++ff) {
    const int f = wave == 0 ? 2 + ff : wave == 1 ? 4 + ff : ff;
    const int ci = wave == 2 ? ff : 0, si = wave == 2 ? 0 : ff;
    f32x4 d0 = {0.f, 0.f, 0.f, 0.f}, d1 = d0;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      d0 = mfma16(b0[si][ks], cf[ci][ks], d0);
      d1 = mfma16(b1[si][ks], cf[ci][ks], d1);
    }
    // elements above the diagonal (s > t) are stored as zeros: the head-per-wave march uses the fragments as they are
    const int f_ti = f == 0 ? 0 : f == 1 ? 1 : f < 4 ? 2 : 3, f_sp = (f == 3 || f == 5) ? 1 : 0;
    const int t_in = 16 * f_ti + lc, s_in = 32 * f_sp + 8 * kq;
    bf16x8 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[r] = s_in + r <= t_in ? (bf16_t)d0[r] : (bf16_t)0.f;
      o[4 + r] = s_in + 4 + r <= t_in ? (bf16_t)d1[r] : (bf16_t)0.f;
    }
    *(bf16x8*)((bf16_t*)a.cb + ((((int64_t)b * a.G + g) * a.nchunks + c) * CB_FRAGS + f) * 512 + lane * 8) = o;
  }
}
// Both parts in one launch: first the blocks of B / C, whose chain is the longer one, then the strips of x
template <int K>
__global__ __launch_bounds__(CONV_THREADS) void conv1d_xbc_cb_kernel(ConvArgs a) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[2][CBQ * CBN];
  const int i = blockIdx.x;
  if (i < a.nbc) conv_bc_cb_block<K>(a, tile, i % a.nchunks, i / a.nchunks, blockIdx.y);
  else conv_xbc_block<bf16_t, K>(a, i - a.nbc, blockIdx.y, a.d_inner);
}

template <typename T, int K>
__global__ void conv1d_update_kernel(const T* __restrict__ x, T* __restrict__ state,
                                     const T* __restrict__ w, const T* __restrict__ bias,
                                     T* __restrict__ y, int C, int silu) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (c >= C) return;
  T* st = state + ((int64_t)b * C + c) * K;
  float acc = bias ? to_f32(bias[c]) : 0.f;
  float win[K];
#pragma unroll
  for (int j = 0; j < K - 1; ++j) win[j] = to_f32(st[j + 1]);
  win[K - 1] = to_f32(x[(int64_t)b * C + c]);
#pragma unroll
  for (int j = 0; j < K; ++j) {
    acc = fmaf(to_f32(w[(int64_t)c * K + j]), win[j], acc);
    st[j] = from_f32<T>(win[j]);
  }
  if (silu) acc = silu_f(acc);
  y[(int64_t)b * C + c] = from_f32<T>(acc);
}

enum { CONV_PLAIN, CONV_XBC, CONV_XBC_CB };
template <typename T, int K>
int launch_conv_k(int form, ConvArgs a, int B, hipStream_t s) {
  constexpr int V = Vec16<T>::N;
  const int c_end = form == CONV_XBC_CB ? a.d_inner : a.C;
  a.nxb = (c_end / V + CONV_THREADS - 1) / CONV_THREADS;
  a.wide = !((uintptr_t)a.w & 15) && !((uintptr_t)a.bias & 15);
  a.per_xcd = ((a.L + CONV_TL - 1) / CONV_TL + 7) / 8;
  a.nchunks = (a.L + CBQ - 1) / CBQ;
  a.nbc = form == CONV_XBC_CB ? a.nchunks * a.G : 0;
  const dim3 grid(a.nbc + 8 * a.nxb * a.per_xcd, B);
  if (form == CONV_PLAIN) conv1d_fwd_kernel<T, K><<<grid, CONV_THREADS, 0, s>>>(a);
  else if (form == CONV_XBC) conv1d_xbc_kernel<T, K><<<grid, CONV_THREADS, 0, s>>>(a);
  else if constexpr (std::is_same<T, bf16_t>::value) conv1d_xbc_cb_kernel<K><<<grid, CONV_THREADS, 0, s>>>(a);
  TV_LAUNCH_CHECK();
}
template <typename T>
int launch_conv(int form, const ConvArgs& a, int B, int K, hipStream_t s) {
  return K == 2 ? launch_conv_k<T, 2>(form, a, B, s) : K == 3 ? launch_conv_k<T, 3>(form, a, B, s) : launch_conv_k<T, 4>(form, a, B, s);
}
int launch_conv_dtype(int form, int dtype, const ConvArgs& a, int B, int K, hipStream_t s, const char* who) {
  switch (dtype) {
    case TV_F32: return launch_conv<float>(form, a, B, K, s);
    case TV_BF16: return launch_conv<bf16_t>(form, a, B, K, s);
    case TV_F16: return launch_conv<f16_t>(form, a, B, K, s);
  }
  TV_UNSUPPORTED("%s: dtype %d", who, dtype);
}

template <typename T>
int launch_conv_update(const void* x, void* st, const void* w, const void* bias, void* y, int B,
                       int C, int K, int silu, hipStream_t s) {
  dim3 grid((C + 255) / 256, B);
#define TV_CONVU_CASE(KK)                                                                  \
  case KK:                                                                                 \
    conv1d_update_kernel<T, KK><<<grid, 256, 0, s>>>((const T*)x, (T*)st, (const T*)w,     \
                                                     (const T*)bias, (T*)y, C, silu);      \
    break;
  switch (K) {
    TV_CONVU_CASE(2)
    TV_CONVU_CASE(3)
    TV_CONVU_CASE(4)
  }
#undef TV_CONVU_CASE
  TV_LAUNCH_CHECK();
}

}  // namespace

extern "C" int tv_causal_conv1d_fwd(const void* x, const void* weight, const void* bias,
                                    const void* halo, void* y, int batch, int seqlen,
                                    int channels, int kernel, int64_t x_stride_b,
                                    int64_t x_stride_l, int64_t y_stride_b, int64_t y_stride_l,
                                    int dtype, int silu, void* stream) {
  TV_CHECK_ARG(weight && (seqlen == 0 || (x && y)), "conv1d: null pointer");   // empty tensors have no storage
  TV_CHECK_ARG(batch > 0 && seqlen >= 0 && channels > 0, "conv1d: bad sizes");
  if (kernel < 2 || kernel > 4) TV_UNSUPPORTED("conv1d: kernel width %d not in [2,4]", kernel);
  if (seqlen == 0) return TV_OK;
  hipStream_t s = (hipStream_t)stream;
  const int vec = dtype == TV_F32 ? 4 : 8;
  if (channels % vec || x_stride_l % vec || y_stride_l % vec || x_stride_b % vec ||
      y_stride_b % vec || ((uintptr_t)x & 15) || ((uintptr_t)y & 15))
    TV_UNSUPPORTED("conv1d: channels/strides/pointers must be 16-byte aligned");
  ConvArgs a{};
  a.x = x; a.w = weight; a.bias = bias; a.halo = halo; a.yx = y;
  a.L = seqlen; a.C = channels; a.silu = silu;
  a.xsb = x_stride_b; a.xsl = x_stride_l; a.ysb = y_stride_b; a.ysl = y_stride_l;
  return launch_conv_dtype(CONV_PLAIN, dtype, a, batch, kernel, s, "conv1d");
}

static int conv1d_xbc_impl(const void* x, const void* weight, const void* bias,
                           const void* halo, void* y_x, void* y_b, void* y_c, void* cb,
                           int batch, int seqlen, int d_inner, int ngroups,
                           int dstate, int kernel, int64_t x_stride_b,
                           int64_t x_stride_l, int dtype, int silu, void* stream, const char* who) {
  TV_CHECK_ARG(weight && (seqlen == 0 || (x && y_x && y_b && y_c)), "%s: null pointer", who);
  TV_CHECK_ARG(batch > 0 && seqlen >= 0 && d_inner > 0 && ngroups > 0 && dstate > 0,
               "%s: bad sizes", who);
  if (kernel < 2 || kernel > 4) TV_UNSUPPORTED("%s: kernel width %d not in [2,4]", who, kernel);
  if (seqlen == 0) return TV_OK;
  const int vec = dtype == TV_F32 ? 4 : 8;
  const int C = d_inner + 2 * ngroups * dstate;
  if (d_inner % vec || dstate % vec || x_stride_l % vec || x_stride_b % vec ||
      ((uintptr_t)x & 15) || ((uintptr_t)y_x & 15) || ((uintptr_t)y_b & 15) || ((uintptr_t)y_c & 15))
    TV_UNSUPPORTED("%s: segments/strides/pointers must be 16-byte aligned", who);
  ConvArgs a{};
  a.x = x; a.w = weight; a.bias = bias; a.halo = halo; a.yx = y_x; a.yb = y_b; a.yc = y_c; a.cb = cb;
  a.L = seqlen; a.C = C; a.d_inner = d_inner; a.G = ngroups; a.N = dstate; a.silu = silu;
  a.xsb = x_stride_b; a.xsl = x_stride_l;
  hipStream_t s = (hipStream_t)stream;
  if (cb) {
    // the scan's C.B^T fragments ride along: the B / C channels of every (chunk, group) are multiplied while they are in LDS
    if (dtype != TV_BF16 || dstate != CBN || ((uintptr_t)cb & 15))
      TV_UNSUPPORTED("%s: the C.B^T output needs bf16 and d_state %d (got dtype %d, N %d)", who, CBN, dtype, dstate);
    return launch_conv<bf16_t>(CONV_XBC_CB, a, batch, kernel, s);
  }
  return launch_conv_dtype(CONV_XBC, dtype, a, batch, kernel, s, who);
}

extern "C" int tv_causal_conv1d_xbc_fwd(const void* x, const void* weight, const void* bias,
                                        const void* halo, void* y_x, void* y_b, void* y_c,
                                        int batch, int seqlen, int d_inner, int ngroups,
                                        int dstate, int kernel, int64_t x_stride_b,
                                        int64_t x_stride_l, int dtype, int silu, void* stream) {
  return conv1d_xbc_impl(x, weight, bias, halo, y_x, y_b, y_c, nullptr, batch, seqlen, d_inner, ngroups, dstate,
                         kernel, x_stride_b, x_stride_l, dtype, silu, stream, "conv1d_xbc");
}

extern "C" size_t tv_ssd_cb_bytes(int batch, int seqlen, int ngroups) {
  if (batch <= 0 || seqlen <= 0 || ngroups <= 0) return 0;
  return (size_t)batch * ngroups * ((seqlen + CBQ - 1) / CBQ) * CB_FRAGS * 512 * sizeof(bf16_t);
}

extern "C" int tv_causal_conv1d_xbc_cb_fwd(const void* x, const void* weight, const void* bias,
                                           const void* halo, void* y_x, void* y_b, void* y_c, void* cb,
                                           int batch, int seqlen, int d_inner, int ngroups,
                                           int dstate, int kernel, int64_t x_stride_b,
                                           int64_t x_stride_l, int dtype, int silu, void* stream) {
  TV_CHECK_ARG(cb || seqlen == 0, "conv1d_xbc_cb: null C.B^T buffer");
  return conv1d_xbc_impl(x, weight, bias, halo, y_x, y_b, y_c, cb, batch, seqlen, d_inner, ngroups, dstate,
                         kernel, x_stride_b, x_stride_l, dtype, silu, stream, "conv1d_xbc_cb");
}

extern "C" int tv_causal_conv1d_update(const void* x, void* conv_state, const void* weight,
                                       const void* bias, void* y, int batch, int channels,
                                       int kernel, int dtype, int silu, void* stream) {
  TV_CHECK_ARG(x && conv_state && weight && y, "conv1d_update: null pointer");
  TV_CHECK_ARG(batch > 0 && channels > 0, "conv1d_update: bad sizes");
  if (kernel < 2 || kernel > 4) TV_UNSUPPORTED("conv1d_update: kernel width %d", kernel);
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case TV_F32:
      return launch_conv_update<float>(x, conv_state, weight, bias, y, batch, channels, kernel,
                                       silu, s);
    case TV_BF16:
      return launch_conv_update<bf16_t>(x, conv_state, weight, bias, y, batch, channels, kernel,
                                        silu, s);
    case TV_F16:
      return launch_conv_update<f16_t>(x, conv_state, weight, bias, y, batch, channels, kernel,
                                       silu, s);
  }
  TV_UNSUPPORTED("conv1d_update: dtype %d", dtype);
}
