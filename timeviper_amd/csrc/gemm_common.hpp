// Shared by the two bf16 GEMM kernels (gemm.hip: one work-group per tile, any shape; gemm_persist.hip: persistent
// work-groups with the tile epilogue hidden in the main loop, the ViT's big shapes).
#pragma once
#include <math.h>
#include <stdlib.h>
#include <type_traits>
#include "ssd_common.hpp"

namespace tvgemm {
using namespace ssdk;

enum { EPI_BIAS = 0, EPI_BIAS_GELU = 1, EPI_ACCUM = 2, EPI_RELU2 = 3, EPI_BIAS_RELU2 = 4, EPI_GLU = 5 };      // EPI_RELU2: of the fp32 sum (moe); EPI_BIAS_RELU2: of the rounded one

constexpr int BM = 256, BN = 256, BK = 64;
constexpr int HALF_BYTES = 128 * BK * 2;          // one half-tile: 128 rows x 128 bytes
constexpr int TILE_BYTES = 4 * HALF_BYTES;        // A0 A1 W0 W1 of one K-tile
constexpr int RING_BYTES = 2 * TILE_BYTES;        // two K-tiles

struct GemmArgs {
  const bf16_t *A, *W;
  const void* bias;        // fp32 or bf16 (bias_f32), may be NULL
  bf16_t* C;
  int M, N, K;
  int64_t lda, ldw, ldc;
  int tiles_m, tiles_n, group_m;
  int bias_f32;
  // grouped products (mixture of experts): the rows [offsets[e], offsets[e + 1]) of C against W + e * w_group; row r of A is
  // row_token[r], or r itself without the list
  const int *offsets, *row_token;
  int groups;
  int64_t w_group;
  // products whose contraction is split over work-groups (tv_gemm_split_fwd): the tiles from `full` on, partial sums [split][tile][256][256]
  float* part;
  int full, splits, relu2;       // relu2: squared ReLU of the rounded sum
  const float* res;        // res_out = res + sum (fp32, rows of N) and C, its bf16 copy, in the sum's place (tv_gemm_split_add_fwd); NULL: none
  float* res_out;
  int ahead;               // gemm_small: all of W asked for once, in order, in front of the loop
};

// same formula as norms.hip's gelu_erf (A&S 7.1.26): the fused and the two-pass path agree bit for bit
__device__ __forceinline__ float gelu_erf_f(float x) {
  // A&S 7.1.26 with 0.5 sqrt(2) folded into the polynomial: gelu(x) = x/2 + |x|/2 erf(|x| / sqrt 2) = x/2 + z (k erf(z)),
  // z = |x| / sqrt 2, k = sqrt(2) / 2 — no copysign, no |x/2| (the packed fp32 forms have no abs modifier), one multiply less
  const float z = fabsf(x) * 0.70710678118654752f;
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f, z, 1.f));
  float p = __builtin_fmaf(0.750526965f, t, -1.02753365f);          // k x {1.061405429, -1.453152027, 1.421413741, -0.284496736, 0.254829592}
  p = __builtin_fmaf(p, t, 1.00509131f);
  p = __builtin_fmaf(p, t, -0.201169565f);
  p = __builtin_fmaf(p, t, 0.180191725f);
  p *= t;
  const float e = __builtin_amdgcn_exp2f(z * z * -1.4426950408889634f);
  const float r = __builtin_fmaf(-p, e, 0.70710678118654752f);       // k erf(z)
  return __builtin_fmaf(z, r, 0.5f * x);
}

#define GEMM_WAIT_VM(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")

// gemm.hip: C = act(gathered A rows . W_e^T) per group on the 256 x 256 tiles; max_rows bounds offsets[groups]
bool grouped_takes(const GemmArgs& a, int64_t max_rows);
int launch_grouped(const GemmArgs& a, int64_t max_rows, int epilogue, hipStream_t st);

// gemm_persist.hip: returns TV_ERR_UNSUPPORTED (without setting the error text) when the shape is not one the persistent
// kernel takes; the caller then runs the per-tile kernel.
bool persist_on();         // not switched off (tv_gemm_set_persist, TV_GEMM_PERSIST=0)
bool persist_takes(const GemmArgs& a, int epilogue);
int launch_persist(const GemmArgs& a, int epilogue, hipStream_t st);
int persist_grid();        // work-groups of the persistent kernels (one per compute unit unless tv_gemm_set_persist says otherwise)

// gemm_drip.hip: persistent 256 x 192 tiles whose finished tile leaves during the next tile's K loop
bool drip_takes(const GemmArgs& a, int epilogue, int grid);
int launch_drip(const GemmArgs& a, int epilogue, int grid, hipStream_t st);

}  // namespace tvgemm
