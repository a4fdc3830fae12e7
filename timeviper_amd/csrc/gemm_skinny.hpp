// What gemm_skinny.hip (products of 2 .. 32 rows on the matrix cores) shares with gemm_mid.hip (33 .. 256 rows: the copies) and with the
// entry points of the matrix-vector kernels (gemv.hip).
#pragma once
#include "ssd_common.hpp"

// 16 bytes a lane: LDS[m0 + 16 lane] = *(sbase + voff), J instructions with the LDS address moving by 1 KiB; NT: non-temporal
template <int J, bool NT>
__device__ __forceinline__ void glds_rows(const void* sbase, const unsigned (&v)[J], unsigned dst) {
  unsigned keep;
#define SK_ONE(NTS, I) "global_load_lds_dwordx4 %" #I ", %5" NTS "\n\t"
#define SK_NEXT "s_add_u32 m0, m0, 1024\n\ts_nop 0\n\t"
#define SK_HEAD "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\ts_nop 0\n\t"
#define SK_ASM(BODY) asm volatile(SK_HEAD BODY "s_mov_b32 m0, %0" : "=&s"(keep) : "v"(v[0]), "v"(v[J > 1 ? 1 : 0]), "v"(v[J > 2 ? 2 : 0]), \
                                  "v"(v[J > 3 ? 3 : 0]), "s"(sbase), "s"(dst) : "memory", "scc")
  if constexpr (NT) {
    if constexpr (J == 1) SK_ASM(SK_ONE(" nt", 1));
    else if constexpr (J == 2) SK_ASM(SK_ONE(" nt", 1) SK_NEXT SK_ONE(" nt", 2));
    else if constexpr (J == 3) SK_ASM(SK_ONE(" nt", 1) SK_NEXT SK_ONE(" nt", 2) SK_NEXT SK_ONE(" nt", 3));
    else SK_ASM(SK_ONE(" nt", 1) SK_NEXT SK_ONE(" nt", 2) SK_NEXT SK_ONE(" nt", 3) SK_NEXT SK_ONE(" nt", 4));
  } else {
    if constexpr (J == 1) SK_ASM(SK_ONE("", 1));
    else if constexpr (J == 2) SK_ASM(SK_ONE("", 1) SK_NEXT SK_ONE("", 2));
    else if constexpr (J == 3) SK_ASM(SK_ONE("", 1) SK_NEXT SK_ONE("", 2) SK_NEXT SK_ONE("", 3));
    else SK_ASM(SK_ONE("", 1) SK_NEXT SK_ONE("", 2) SK_NEXT SK_ONE("", 3) SK_NEXT SK_ONE("", 4));
  }
#undef SK_ASM
#undef SK_HEAD
#undef SK_NEXT
#undef SK_ONE
}

// far_rows: how far behind a work-group's first row of W its last one may lie, beside the 32 of its share
bool tv_skinny_takes(const void* x, const void* W, int M, int K, int64_t xs, int64_t ldw, int64_t far_rows);
int tv_skinny_add(const void* x, const void* W, const void* bias, const float* residual, float* residual_out, void* h_out, int M, int N, int K,
                  int64_t xs, int64_t ldw, hipStream_t st);
int tv_skinny_pair(const void* x, const void* x2, const void* W, const void* bias, void* y, void* act, int M, int n1, int ff, int K,
                   int64_t xs, int64_t x2s, int64_t ldw, int64_t ys, int64_t as, hipStream_t st);
