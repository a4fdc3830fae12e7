// Products of 2 .. 32 rows on the matrix cores (gemm_skinny.hip), for the entry points of the matrix-vector kernels (gemv.hip).
#pragma once
#include "ssd_common.hpp"

// far_rows: how far behind a work-group's first row of W its last one may lie, beside the 32 of its share
bool tv_skinny_takes(const void* x, const void* W, int M, int K, int64_t xs, int64_t ldw, int64_t far_rows);
int tv_skinny_add(const void* x, const void* W, const void* bias, const float* residual, float* residual_out, void* h_out, int M, int N, int K,
                  int64_t xs, int64_t ldw, hipStream_t st);
int tv_skinny_pair(const void* x, const void* x2, const void* W, const void* bias, void* y, void* act, int M, int n1, int ff, int K,
                   int64_t xs, int64_t x2s, int64_t ldw, int64_t ys, int64_t as, hipStream_t st);
