// Mixture of experts for single tokens (decode, bf16): two launches that stream the chosen experts' matrices once.
//   tv_moe_decode_up    choice of the experts from the router's logits (softmax, correction, top), then
//                       u[c] = relu(W_up[e_c] h)^2 for the choices c of every token; ids / weights are written for the second launch
//   tv_moe_decode_down  y = sum_c w_c W_down[e_c] u[c] + sum over identity choices w_c x
// Matrix-vector products: HBM-bound, a row of W per wave, 16-byte non-temporal loads, two rows in flight.
#include "moe.hpp"

namespace tvmoe {
namespace {

constexpr int MD_THREADS = 256, MD_WAVES = 4;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot8(bf16x8 a, bf16x8 b, float acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    acc = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{a[2 * j], a[2 * j + 1]}, bf16x2{b[2 * j], b[2 * j + 1]}, acc, false);
  return acc;
}
__device__ __forceinline__ bf16x8 ldw(const bf16_t* p) { return __builtin_nontemporal_load((const bf16x8*)p); }

struct MdArgs {
  const float *logits, *x;       // (M, E + identity), (M, D)
  const bf16_t *corr, *h, *up, *down;
  bf16_t *u, *y;                 // (M * top, ff), (M, D)
  int* ids;                      // (M, top)
  float* wts;
  int E, n_out, top, D, ff;
};

// NB: 64-piece load instructions of a row (D <= 512 NB); ME: router outputs at most
template <int NB, int ME>
__global__ __launch_bounds__(MD_THREADS) void moe_decode_up_kernel(MdArgs a) {
  __shared__ __attribute__((aligned(16))) float sz[ME], sc[ME];
  __shared__ int pick;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = blockIdx.y, t = c / a.top, k = c % a.top;
  const int nv = a.D / 8;
  bf16x8 hx[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const bf16x8 z = {};
    const int p = 64 * i + lane;
    hx[i] = p < nv ? *(const bf16x8*)(a.h + (int64_t)t * a.D + 8 * p) : z;
  }
  if (wave == 0) {
    for (int e = lane; e < a.n_out; e += 64) sz[e] = a.logits[(int64_t)t * a.n_out + e];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    select_experts<bf16_t, ME>(sz, sc, a.corr, a.n_out, a.top, lane, [&](int p, int e, float s) {
      if (p == k) {
        pick = e;
        if (blockIdx.x == 0) {
          a.ids[c] = e;
          a.wts[c] = s;
        }
      }
    });
  }
  __syncthreads();
  const int e = pick;
  if (e >= a.E) return;                        // an identity expert
  const bf16_t* W = a.up + (int64_t)e * a.ff * a.D;
  const int stride = gridDim.x * MD_WAVES;
  for (int n = blockIdx.x * MD_WAVES + wave; n < a.ff; n += 2 * stride) {
    const bool two = n + stride < a.ff;
    bf16x8 w0[NB], w1[NB];
    const bf16_t *r0 = W + (int64_t)n * a.D + 8 * lane, *r1 = two ? r0 + (int64_t)stride * a.D : r0;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const bf16x8 z = {};
      const bool in = 64 * i + lane < nv;
      w0[i] = in ? ldw(r0 + 512 * i) : z;
      w1[i] = in && two ? ldw(r1 + 512 * i) : z;
    }
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      s0 = dot8(w0[i], hx[i], s0);
      s1 = dot8(w1[i], hx[i], s1);
    }
    s0 = fmaxf(wave_sum_dpp(s0), 0.f);
    s1 = fmaxf(wave_sum_dpp(s1), 0.f);
    if (lane == 0) {
      a.u[(int64_t)c * a.ff + n] = (bf16_t)(s0 * s0);
      if (two) a.u[(int64_t)c * a.ff + n + stride] = (bf16_t)(s1 * s1);
    }
  }
}

__global__ __launch_bounds__(MD_THREADS) void moe_decode_down_kernel(MdArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char md_smem[];
  __shared__ int rows[MOE_MAX_TOP];
  __shared__ float wr[MOE_MAX_TOP], ident;
  __shared__ int nrow;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = blockIdx.y, pf = a.ff / 8;
  bf16_t* su = (bf16_t*)md_smem;               // u of the choices that have matrices, one after the other
  if (tid == 0) {
    int n = 0;
    float id = 0.f;
    for (int k = 0; k < a.top; ++k) {
      const int e = a.ids[t * a.top + k];
      const float w = a.wts[t * a.top + k];
      if (e < a.E) {
        rows[n] = e | k << 16;
        wr[n++] = w;
      } else {
        id += w;
      }
    }
    nrow = n;
    ident = id;
  }
  __syncthreads();
  const int nr = nrow, P = nr * pf;            // 16-byte pieces of a row of the stacked matrices
  for (int p = tid; p < P; p += MD_THREADS) {
    const int c = p / pf;
    *(bf16x8*)(su + 8 * p) = *(const bf16x8*)(a.u + ((int64_t)t * a.top + (rows[c] >> 16)) * a.ff + 8 * (p - c * pf));
  }
  __syncthreads();
  constexpr int NB = 8;
  const int stride = gridDim.x * MD_WAVES;
  for (int n = blockIdx.x * MD_WAVES + wave; n < a.D; n += 2 * stride) {
    const bool two = n + stride < a.D;
    float s0 = 0.f, s1 = 0.f;
    for (int p0 = 0; p0 < P; p0 += 64 * NB) {
      bf16x8 w0[NB], w1[NB];
      float wt[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int p = p0 + 64 * i + lane;
        const bf16x8 z = {};
        const bool in = p < P;
        const int c = in ? p / pf : 0;
        const bf16_t* r = a.down + ((int64_t)(rows[c] & 0xffff) * a.D + n) * a.ff + 8 * (p - c * pf);
        w0[i] = in ? ldw(r) : z;
        w1[i] = in && two ? ldw(r + (int64_t)stride * a.ff) : z;
        wt[i] = wr[c];
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int p = p0 + 64 * i + lane;
        if (p < P) {
          const bf16x8 uv = *(const bf16x8*)(su + 8 * p);
          s0 = fmaf(wt[i], dot8(w0[i], uv, 0.f), s0);
          s1 = fmaf(wt[i], dot8(w1[i], uv, 0.f), s1);
        }
      }
    }
    s0 = wave_sum_dpp(s0);
    s1 = wave_sum_dpp(s1);
    if (lane == 0) {
      a.y[(int64_t)t * a.D + n] = (bf16_t)fmaf(ident, a.x[(int64_t)t * a.D + n], s0);
      if (two) a.y[(int64_t)t * a.D + n + stride] = (bf16_t)fmaf(ident, a.x[(int64_t)t * a.D + n + stride], s1);
    }
  }
}

}  // namespace
}  // namespace tvmoe

using namespace tvmoe;

extern "C" int tv_moe_decode_fwd(const float* logits, const void* correction, const void* h, const float* x, const void* up,
                                 const void* down, int* ids, float* weights, void* u, void* y, int tokens, int experts, int n_out,
                                 int top, int D, int ff, void* stream) {
  TV_CHECK_ARG(logits && h && x && up && down && ids && weights && u && y, "moe_decode: null pointer");
  TV_CHECK_ARG(tokens > 0 && tokens <= 64 && experts > 0 && n_out >= experts && top > 0 && top <= n_out && D > 0 && ff > 0, "moe_decode: bad sizes");
  if (n_out > 256 || top > MOE_MAX_TOP || experts >= 65536 || D % 8 || ff % 8 || D > 8192 || (size_t)top * ff * 2 > 128 * 1024 ||
      ((uintptr_t)h & 15) || ((uintptr_t)up & 15) || ((uintptr_t)down & 15) || ((uintptr_t)u & 15))
    TV_UNSUPPORTED("moe_decode: %d outputs (<= 256), top %d (<= %d), width %d and ff %d multiples of 8, width <= 8192, top x ff <= 65536",
                   n_out, top, MOE_MAX_TOP, D, ff);
  MdArgs a{logits, x, (const bf16_t*)correction, (const bf16_t*)h, (const bf16_t*)up, (const bf16_t*)down, (bf16_t*)u, (bf16_t*)y, ids, weights,
           experts, n_out, top, D, ff};
  hipStream_t st = (hipStream_t)stream;
  // about two work-groups a compute unit over all choices; at least two rows a wave
  auto wgs = [&](int rows, int groups) {
    int w = (2 * tv_cu_count() + groups - 1) / groups;
    const int most = (rows + 2 * MD_WAVES - 1) / (2 * MD_WAVES);
    if (w > most) w = most;
    return w < 1 ? 1 : w;
  };
  const dim3 g1((unsigned)wgs(ff, tokens * top), (unsigned)(tokens * top));
#define MOE_UP(NB)                                                              \
  do {                                                                          \
    if (n_out <= 128) moe_decode_up_kernel<NB, 128><<<g1, MD_THREADS, 0, st>>>(a); \
    else moe_decode_up_kernel<NB, 256><<<g1, MD_THREADS, 0, st>>>(a);           \
  } while (0)
  if (D <= 2048) MOE_UP(4);
  else if (D <= 4096) MOE_UP(8);
  else MOE_UP(16);
#undef MOE_UP
  const size_t lds = (size_t)top * ff * sizeof(bf16_t);
  static const hipError_t attr = hipFuncSetAttribute((const void*)moe_decode_down_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
  if (attr != hipSuccess) {
    tv_set_error("moe_decode: cannot reserve 128 KiB of LDS: %s", hipGetErrorString(attr));
    return TV_ERR_LAUNCH;
  }
  moe_decode_down_kernel<<<dim3((unsigned)wgs(D, tokens), (unsigned)tokens), MD_THREADS, lds, st>>>(a);
  TV_LAUNCH_CHECK();
}
