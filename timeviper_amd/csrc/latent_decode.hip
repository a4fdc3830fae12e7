// Latent attention of a decode step on the matrix cores (bf16, latents of up to 512 dimensions): four launches.
//
//   latent_prep_kernel    q~[b][h][r] = sum_d q[b][h][d] W_uk[h dim + d][r] (the query taken to the latents), and the norm of the
//                         step's own latents with their way into the cache
//   latent_split_kernel   softmax(q~ . c) c over the cached latents: ONE shared "key / value head" of `rank` dimensions for all
//                         query heads, the keys split over work-groups.  Per tile of 32 latents (copied to LDS once, used twice):
//                           S^T[key][head] = C . Q~^T      A = latent rows, B = query fragments held in registers
//                           O^T[r][head]  += C^T . P^T     A = the same tile read transposed, B = the weights
//                         two waves score the tile's two 16-key groups (per block of 16 heads), every wave owns a quarter of the
//                         latent dimensions of O
//   latent_merge_kernel   merges the splits' (maximum, sum, O) with the head's sink, 64 latent dimensions a work-group
//   latent_out_kernel     multiplies with W_uv
//
// LDS: 16-byte chunk c of row k lies at chunk c ^ f(k) (f: a permutation of 0 .. 15 over 16 rows): row reads and transposing
// reads are both conflict-free.  Latent sizes between the tile sizes are padded with zeros that are written once.
#include "ssd_common.hpp"

namespace {
using namespace ssdk;

constexpr int LD_THREADS = 256, LD_TILE = 32, LD_PS = 80;      // LD_PS: bytes between two heads' weights of a tile
typedef __attribute__((address_space(3))) bf16x4 ld_lds4;
typedef __attribute__((address_space(3))) const bf16x8 ld_lds8;

struct LdArgs {
  const bf16_t *q, *uk, *uv, *c_new, *c_norm;
  bf16_t *lat, *qt, *o;
  const float* sink;
  float *part_o, *part_ml, *ol;          // ol [B][H][R]: the weighted latents
  const int *rows, *keys, *slot;
  int B, H, dim, vdim, R, nsplit;
  int64_t qs, cs, os, slot_stride;       // row strides of q, c_new, o; elements between two slots
  float scale_log2, eps;
};

__device__ __forceinline__ unsigned swz(int row) { return (unsigned)(((row & 3) << 1) | (row & 8) | ((row >> 2) & 1)); }
__device__ __forceinline__ f32x4 mm(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

__global__ __launch_bounds__(LD_THREADS) void latent_prep_kernel(LdArgs a) {
  __shared__ float sh[16][128 + 4];
  __shared__ float red[4];
  const int tid = threadIdx.x, h = blockIdx.y, b = blockIdx.z;
  if (h == a.H) {                          // the step's own latent of sequence b: norm, into the cache
    if (blockIdx.x) return;
    const bf16_t* c = a.c_new + (int64_t)b * a.cs;
    float ssq = 0.f;
    for (int r = tid; r < a.R; r += LD_THREADS) ssq = fmaf((float)c[r], (float)c[r], ssq);
    ssq = wave_sum(ssq);
    if ((tid & 63) == 0) red[tid >> 6] = ssq;
    __syncthreads();
    const float rstd = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)a.R + a.eps);
    bf16_t* dst = a.lat + (int64_t)a.rows[b] * a.R;
    for (int r = tid; r < a.R; r += LD_THREADS) dst[r] = (bf16_t)((float)c[r] * rstd * (float)a.c_norm[r]);
    return;
  }
  const int g = tid >> 4, r0 = blockIdx.x * 128 + 8 * (tid & 15);      // 16 groups of d, 8 latent dims a thread
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (r0 < a.R) {
    const bf16_t* qh = a.q + (int64_t)b * a.qs + (int64_t)h * a.dim;
    const bf16_t* w = a.uk + (int64_t)h * a.dim * a.R + r0;
#pragma unroll 8
    for (int d = g; d < a.dim; d += 16) {
      const bf16x8 v = *(const bf16x8*)(w + (int64_t)d * a.R);
      const float qd = (float)qh[d];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = fmaf(qd, (float)v[i], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) sh[g][8 * (tid & 15) + i] = acc[i];
  __syncthreads();
  if (tid < 128 && blockIdx.x * 128 + tid < a.R) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) s += sh[j][tid];
    a.qt[((int64_t)b * a.H + h) * a.R + blockIdx.x * 128 + tid] = (bf16_t)s;
  }
}

// keys [split * chunk, ...) of a sequence with n keys; chunk is a multiple of the tile
__device__ __forceinline__ int split_chunk(int n, int nsplit) {
  const int per = (n + nsplit - 1) / nsplit;
  return max((per + LD_TILE - 1) / LD_TILE * LD_TILE, LD_TILE);
}

// RP: padded latent size, HB: blocks of 16 heads a work-group takes
template <int RP, int HB>
__global__ __launch_bounds__(LD_THREADS) void latent_split_kernel(LdArgs a) {
  constexpr int KS = RP / 32, RT = RP / 64;          // k-steps of the scores; 16-dim tiles of O per wave
  constexpr unsigned ROWB = RP * 2, STAGE = LD_TILE * ROWB, P0 = 2 * STAGE, M0 = P0 + HB * 16 * LD_PS;
  constexpr int RPI = 1024 / ROWB;                   // rows one copy instruction covers
  constexpr int CP = LD_TILE / RPI / 4;              // copy instructions per wave and tile
  extern __shared__ __attribute__((aligned(16))) unsigned char ld_smem[];
  const unsigned lds = lds_addr_of(ld_smem);
  float* sm = (float*)(ld_smem + M0);                // [HB][2][16]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, kq = lane >> 4;
  const int split = blockIdx.x, b = blockIdx.z, head0 = blockIdx.y * 16 * HB;
  const int n = a.keys[b], chunk = split_chunk(n, a.nsplit);
  const int k0 = split * chunk, k1 = min(n, k0 + chunk);
  if (k0 >= k1) return;                              // (the merge skips the same splits)
  const int ntile = (k1 - k0 + LD_TILE - 1) / LD_TILE, last = k1 - k0 - 1;
  const bf16_t* base = a.lat + (int64_t)a.slot[b] * a.slot_stride + (int64_t)k0 * a.R;

  if (a.R < RP) {                                    // padding: zeros, never copied over
    const bf16x8 z = {};
    for (unsigned i = 16 * tid; i < 2 * STAGE; i += 16 * LD_THREADS) *(bf16x8*)(ld_smem + i) = z;
    __syncthreads();
  }
  const int nchunk = a.R / 8;
  auto copy_tile = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const int row = RPI * (wave * CP + i) + lane / (64 / RPI);
      const unsigned ch = (unsigned)(lane % (64 / RPI)) ^ swz(row & 15);
      const int key = min(LD_TILE * t + row, last);  // rows past the range repeat its last key (masked)
      const unsigned dst = lds + (unsigned)(t & 1) * STAGE + (unsigned)(wave * CP + i) * 1024u;
      if ((int)ch < nchunk) glds16(uniform_ptr(base), (unsigned)key * (unsigned)(a.R * 2) + 16u * ch, dst);
    }
  };
  // scoring role: key group of 16, block of heads
  const int kg = wave & 1, hb = HB == 2 ? wave >> 1 : 0;
  const bool scores = HB == 2 || wave < 2;
  bf16x8 qf[KS];
  {
    const int h = head0 + 16 * hb + lc;
    const bf16_t* qp = a.qt + ((int64_t)b * a.H + min(h, a.H - 1)) * a.R;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 z = {};
      const int r = 32 * ks + 8 * kq;
      qf[ks] = scores && h < a.H && r < a.R ? *(const bf16x8*)(qp + r) : z;
    }
  }
  f32x4 O[HB][RT];
#pragma unroll
  for (int j = 0; j < HB; ++j)
#pragma unroll
    for (int r = 0; r < RT; ++r) O[j][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[HB], l_run = 0.f;
#pragma unroll
  for (int j = 0; j < HB; ++j) m_run[j] = -INFINITY;
  copy_tile(0);
  for (int t = 0; t < ntile; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                                 // tile t is there; nobody reads tile t - 1 any more
    if (t + 1 < ntile) copy_tile(t + 1);
    const unsigned st = lds + (unsigned)(t & 1) * STAGE;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (scores) {
      const int row = 16 * kg + lc;
      const unsigned ra = st + (unsigned)row * ROWB;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = mm(*(ld_lds8*)(size_t)(ra + (((unsigned)(4 * ks + kq) ^ swz(row & 15)) << 4)), qf[ks], s);
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[r] = LD_TILE * t + 16 * kg + 4 * kq + r <= last ? s[r] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, s[r]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      if (kq == 0) sm[(hb * 2 + kg) * 16 + lc] = mx;
    }
    __syncthreads();
    float alpha[HB];
#pragma unroll
    for (int j = 0; j < HB; ++j) {
      const float m_new = fmaxf(m_run[j], fmaxf(sm[(j * 2) * 16 + lc], sm[(j * 2 + 1) * 16 + lc]));      // finite: group 0 holds a key
      alpha[j] = __builtin_amdgcn_exp2f(m_run[j] - m_new);
      m_run[j] = m_new;
    }
    if (scores) {
      const float m = HB == 2 && hb ? m_run[HB - 1] : m_run[0], al = HB == 2 && hb ? alpha[HB - 1] : alpha[0];
      bf16x4 p;
      float ps = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(s[r] - m);
        ps += e;
        p[r] = (bf16_t)e;
      }
      l_run = l_run * al + ps;
      *(bf16x4*)(ld_smem + P0 + (unsigned)(16 * hb + lc) * LD_PS + 2u * (16 * kg + 4 * kq)) = p;
    }
    __syncthreads();
    bf16x8 pf[HB];
#pragma unroll
    for (int j = 0; j < HB; ++j) pf[j] = *(ld_lds8*)(size_t)(lds + P0 + (unsigned)(16 * j + lc) * LD_PS + 16u * kq);
    const int row = 8 * kq + (lc >> 2);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const unsigned ch = (unsigned)(2 * (wave * RT + rt) + ((lc & 3) >> 1));
      const unsigned half = 8u * (lc & 1);
      const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ld_lds4*)(size_t)(st + (unsigned)row * ROWB + ((ch ^ swz(row & 15)) << 4) + half));
      const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((ld_lds4*)(size_t)(st + (unsigned)(row + 4) * ROWB + ((ch ^ swz((row + 4) & 15)) << 4) + half));
      const bf16x8 cf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int j = 0; j < HB; ++j) {
        O[j][rt] *= alpha[j];
        O[j][rt] = mm(cf, pf[j], O[j][rt]);
      }
    }
  }
  // ---- partial results: O^T rows r = 16 tile + 4 kq + 0..3 of head lc
#pragma unroll
  for (int j = 0; j < HB; ++j) {
    const int h = head0 + 16 * j + lc;
    if (h < a.H) {
      float* po = a.part_o + (((int64_t)b * a.H + h) * a.nsplit + split) * a.R;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int r = 16 * (wave * RT + rt) + 4 * kq;
        if (r < a.R) *(f32x4*)(po + r) = O[j][rt];
      }
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  __syncthreads();                                   // the maxima have been read
  if (scores && kq == 0) sm[(hb * 2 + kg) * 16 + lc] = l_run;
  __syncthreads();
  if (wave == 0 && kq == 0) {
#pragma unroll
    for (int j = 0; j < HB; ++j) {
      const int h = head0 + 16 * j + lc;
      if (h < a.H) {
        float* ml = a.part_ml + (((int64_t)b * a.H + h) * a.nsplit + split) * 2;
        ml[0] = m_run[j];
        ml[1] = sm[(j * 2) * 16 + lc] + sm[(j * 2 + 1) * 16 + lc];
      }
    }
  }
}

constexpr int LD_MAXSPLIT = 256, LD_VB = 32;

__global__ __launch_bounds__(LD_THREADS) void latent_merge_kernel(LdArgs a) {
  __shared__ float sw[LD_MAXSPLIT], red[4];
  __shared__ f32x4 so[16][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = blockIdx.y, b = blockIdx.z;
  const int n = a.keys[b], chunk = split_chunk(n, a.nsplit), nv = (n + chunk - 1) / chunk;
  const int64_t s0 = ((int64_t)b * a.H + h) * a.nsplit;
  const float sink2 = a.sink[h] * 1.4426950408889634f;
  float ms = -INFINITY, ls = 0.f;
  if (tid < nv) {
    ms = a.part_ml[(s0 + tid) * 2];
    ls = a.part_ml[(s0 + tid) * 2 + 1];
  }
  const float wm = wave_max(ms);
  if (lane == 0) red[wave] = wm;
  __syncthreads();
  const float M = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), sink2);
  __syncthreads();
  const float w = __builtin_amdgcn_exp2f(ms - M);    // (no split: 2^-inf)
  sw[tid] = w;
  const float wl = wave_sum(w * ls);
  if (lane == 0) red[wave] = wl;
  __syncthreads();
  const float inv = 1.f / (red[0] + red[1] + red[2] + red[3] + __builtin_amdgcn_exp2f(sink2 - M));
  // 16 four-dim columns x 16 groups of splits
  const int col = tid & 15, g = tid >> 4, r = blockIdx.x * 64 + 4 * col;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (r < a.R) {
    const float* po = a.part_o + s0 * a.R + r;
    constexpr int U = 8;
    for (int s = g; s < nv; s += 16 * U) {
      f32x4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = *(const f32x4*)(po + (int64_t)min(s + 16 * u, nv - 1) * a.R);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float ww = s + 16 * u < nv ? sw[s + 16 * u] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(ww, v[u][i], acc[i]);
      }
    }
  }
  so[g][col] = acc;
  __syncthreads();
  if (tid < 64 && blockIdx.x * 64 + tid < a.R) {
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) t += so[j][tid >> 2][tid & 3];
    a.ol[((int64_t)b * a.H + h) * a.R + blockIdx.x * 64 + tid] = t * inv;
  }
}

__global__ __launch_bounds__(LD_THREADS) void latent_out_kernel(LdArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = blockIdx.y, b = blockIdx.z;
  constexpr int RW = LD_VB / 4;
  const bool in = 8 * lane < a.R;
  bf16x8 wv[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int v = blockIdx.x * LD_VB + 4 * i + wave;
    const bf16x8 z = {};
    wv[i] = in && v < a.vdim ? *(const bf16x8*)(a.uv + ((int64_t)h * a.vdim + v) * a.R + 8 * lane) : z;
  }
  float x[8];
  const float* ol = a.ol + ((int64_t)b * a.H + h) * a.R + 8 * lane;
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = in ? ol[i] : 0.f;
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int v = blockIdx.x * LD_VB + 4 * i + wave;
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s = fmaf(x[j], (float)wv[i][j], s);
    s = wave_sum_dpp(s);
    if (lane == 0 && v < a.vdim) a.o[(int64_t)b * a.os + (int64_t)h * a.vdim + v] = (bf16_t)s;
  }
}

int pick_splits(int batch, int groups, int capacity) {
  int want = (2 * tv_cu_count() + batch * groups - 1) / (batch * groups);       // two work-groups a compute unit
  const int most = (capacity + 2 * LD_TILE - 1) / (2 * LD_TILE);             // of at least two tiles: a split writes 2 H R floats
  if (want > most) want = most;
  if (want > LD_MAXSPLIT) want = LD_MAXSPLIT;
  return want < 1 ? 1 : want;
}

template <int RP, int HB>
int launch_split(const LdArgs& a, hipStream_t st) {
  constexpr int lds = 2 * LD_TILE * RP * 2 + HB * 16 * LD_PS + HB * 2 * 16 * 4;
  static const hipError_t attr = hipFuncSetAttribute((const void*)latent_split_kernel<RP, HB>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) {
    tv_set_error("latent_decode: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  latent_split_kernel<RP, HB><<<dim3((unsigned)a.nsplit, (unsigned)((a.H + 16 * HB - 1) / (16 * HB)), (unsigned)a.B), LD_THREADS, lds, st>>>(a);
  return TV_OK;
}

}  // namespace

extern "C" size_t tv_latent_decode_workspace_bytes(int batch, int nheads, int rank, int capacity) {
  if (batch <= 0 || nheads <= 0 || rank <= 0 || capacity <= 0) return 0;
  const int groups = nheads > 16 ? (nheads + 31) / 32 : 1;
  const size_t ns = (size_t)pick_splits(batch, groups, capacity), bh = (size_t)batch * nheads;
  return bh * ns * rank * 4 + bh * ns * 8 + bh * rank * 6 + 64;
}

extern "C" int tv_latent_decode_fwd(const void* q, const void* w_uk, const void* w_uv, void* latents, const void* c_new,
                                    const void* c_norm, float eps, const int* rows, const int* keys, const int* slot,
                                    const float* sink, void* o, int batch, int nheads, int dim, int vdim, int rank, int capacity,
                                    int64_t q_stride, int64_t c_stride, int64_t o_stride, float scale, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(q && w_uk && w_uv && latents && keys && slot && sink && o && (!c_new || (c_norm && rows)), "latent_decode: null pointer");
  TV_CHECK_ARG(batch > 0 && batch < 65536 && nheads > 0 && nheads < 65535 && dim > 0 && vdim > 0 && rank > 0 && capacity > 0 && scale > 0.f,
               "latent_decode: bad sizes (or non-positive scale)");
  if (rank % 8 || rank > 512 || ((uintptr_t)w_uk & 15) || ((uintptr_t)w_uv & 15) || ((uintptr_t)latents & 15) ||
      (int64_t)capacity * rank * 2 >= (1ll << 32))
    TV_UNSUPPORTED("latent_decode: latents of %d dimensions (a multiple of 8, at most 512), 16-byte aligned operands", rank);
  const int groups = nheads > 16 ? (nheads + 31) / 32 : 1;
  const size_t need = tv_latent_decode_workspace_bytes(batch, nheads, rank, capacity);
  TV_CHECK_ARG(workspace && workspace_bytes >= need && ((uintptr_t)workspace & 15) == 0, "latent_decode: workspace of %zu bytes needed, got %zu",
               need, workspace_bytes);
  LdArgs a{};
  a.q = (const bf16_t*)q; a.uk = (const bf16_t*)w_uk; a.uv = (const bf16_t*)w_uv; a.c_new = (const bf16_t*)c_new; a.c_norm = (const bf16_t*)c_norm;
  a.lat = (bf16_t*)latents; a.o = (bf16_t*)o; a.sink = sink; a.rows = rows; a.keys = keys; a.slot = slot;
  a.B = batch; a.H = nheads; a.dim = dim; a.vdim = vdim; a.R = rank; a.nsplit = pick_splits(batch, groups, capacity);
  a.qs = q_stride; a.cs = c_stride; a.os = o_stride; a.slot_stride = (int64_t)capacity * rank;
  a.scale_log2 = scale * 1.4426950408889634f; a.eps = eps;
  const size_t bh = (size_t)batch * nheads;
  a.part_o = (float*)workspace;
  a.part_ml = a.part_o + bh * a.nsplit * rank;
  a.ol = (float*)(((uintptr_t)(a.part_ml + bh * a.nsplit * 2) + 15) & ~(uintptr_t)15);
  a.qt = (bf16_t*)(a.ol + bh * rank);
  hipStream_t st = (hipStream_t)stream;
  latent_prep_kernel<<<dim3((unsigned)((rank + 127) / 128), (unsigned)(nheads + (c_new ? 1 : 0)), (unsigned)batch), LD_THREADS, 0, st>>>(a);
  int e;
  if (rank <= 128) e = groups == 1 && nheads <= 16 ? launch_split<128, 1>(a, st) : launch_split<128, 2>(a, st);
  else if (rank <= 256) e = nheads <= 16 ? launch_split<256, 1>(a, st) : launch_split<256, 2>(a, st);
  else e = nheads <= 16 ? launch_split<512, 1>(a, st) : launch_split<512, 2>(a, st);
  if (e != TV_OK) return e;
  latent_merge_kernel<<<dim3((unsigned)((rank + 63) / 64), (unsigned)nheads, (unsigned)batch), LD_THREADS, 0, st>>>(a);
  latent_out_kernel<<<dim3((unsigned)((vdim + LD_VB - 1) / LD_VB), (unsigned)nheads, (unsigned)batch), LD_THREADS, 0, st>>>(a);
  TV_LAUNCH_CHECK();
}
