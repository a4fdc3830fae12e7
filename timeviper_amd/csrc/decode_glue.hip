// What stands between the layers of a decoded token and the next one: the new keys and values into the cache, the counters, the greedy choice.
// A launch of these takes 4 - 5 us however little it does, so what counts is how many there are, and how many compute units read the logits.
// Measured (one sequence, in a replayed graph): index_copy_ twice 9.2 -> 4.7 us, += 1 twice 8.4 -> 3.9, argmax of 131 072 logits (one work-group
// a row) 12.8 -> 4.8 + 4.6; a token 433 -> 421 us with the gaps that went.  The counters in the greedy
// choice's last launch, and the logits as fp32 with their norm out of the product (gemv.hip): 420 -> 413 (three launches of 4 - 5 us when traced alone).
#include <mutex>

#include "common.hpp"

namespace {

// sequence blockIdx.x, K (y 0) or V (y 1): one row of 16-byte pieces to position *pos of the cache; a position outside it writes nothing
__global__ __launch_bounds__(256) void kv_append_kernel(const uint4* __restrict__ k, const uint4* __restrict__ v, uint4* __restrict__ kb,
                                                        uint4* __restrict__ vb, const int64_t* __restrict__ pos, int64_t capacity, int pieces,
                                                        int64_t ksb, int64_t vsb, int64_t kbb, int64_t kbl, int64_t vbb, int64_t vbl) {
  const int64_t t = *pos;
  if (t < 0 || t >= capacity) return;
  const bool second = blockIdx.y != 0;
  const uint4* src = second ? v + blockIdx.x * vsb : k + blockIdx.x * ksb;
  uint4* dst = second ? vb + blockIdx.x * vbb + t * vbl : kb + blockIdx.x * kbb + t * kbl;
  for (int i = threadIdx.x; i < pieces; i += 256) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void count_up_kernel(int64_t* __restrict__ pos, int* __restrict__ lens, int n) {
  if (threadIdx.x == 0) pos[0] += 1;
  for (int i = threadIdx.x; i < n; i += 256) lens[i] += 1;
}

// the larger of two (value, position): NaN above all, the lower position of equals (torch.argmax)
struct Best {
  float v;
  unsigned i;
};
__device__ __forceinline__ Best better(Best a, Best b) {
  const bool an = a.v != a.v, bn = b.v != b.v;
  const bool b_wins = an != bn ? bn : (!an && a.v != b.v) ? b.v > a.v : b.i < a.i;
  return b_wins ? b : a;
}
__device__ __forceinline__ Best wave_best(Best x) {
#pragma unroll
  for (int o = 32; o; o >>= 1) x = better(x, Best{__shfl_xor(x.v, o), (unsigned)__shfl_xor((int)x.i, o)});
  return x;
}
__device__ __forceinline__ Best nothing() { return Best{-__builtin_inff(), 0xffffffffu}; }

constexpr int ARG_BLOCKS = 64;
// row blockIdx.y, share blockIdx.x of its elements
__global__ __launch_bounds__(256) void argmax_part_kernel(const float* __restrict__ x, Best* __restrict__ part, int n, int64_t stride, int wide) {
  const float* row = x + blockIdx.y * stride;
  const int share = ((n + ARG_BLOCKS - 1) / ARG_BLOCKS + 3) & ~3, lo = blockIdx.x * share, hi = min(n, lo + share);
  Best b = nothing();
  if (wide) {
    for (int i = lo + 4 * threadIdx.x; i < hi; i += 1024) {
      const f32x4 v = *(const f32x4*)(row + i);                // (n % 4 == 0: whole pieces)
#pragma unroll
      for (int j = 0; j < 4; ++j) b = better(b, Best{v[j], (unsigned)(i + j)});
    }
  } else {
    for (int i = lo + threadIdx.x; i < hi; i += 256) b = better(b, Best{row[i], (unsigned)i});
  }
  b = wave_best(b);
  __shared__ Best s[4];
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = b;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.y * ARG_BLOCKS + blockIdx.x] = better(better(s[0], s[1]), better(s[2], s[3]));
}
// ... and the counters that count_up_kernel moves (either may be NULL), by the first row's work-group (3.9 us as a launch of its own)
__global__ __launch_bounds__(ARG_BLOCKS) void argmax_rows_kernel(const Best* __restrict__ part, int64_t* __restrict__ out, int64_t* __restrict__ pos,
                                                                 int* __restrict__ lens, int nlens) {
  const Best b = wave_best(part[blockIdx.x * ARG_BLOCKS + threadIdx.x]);
  if (threadIdx.x == 0) out[blockIdx.x] = (int64_t)b.i;
  if (blockIdx.x == 0) {
    if (pos && threadIdx.x == 0) pos[0] += 1;
    if (lens)
      for (int i = threadIdx.x; i < nlens; i += ARG_BLOCKS) lens[i] += 1;
  }
}

// Where the rows of a packed step live, from host numbers that ride in the launch: sequence blockIdx.y of up to PLAN_SEQ, its share blockIdx.x
// of the rows.  Copied from pageable memory instead, each of the five arrays waited for the device to run dry: 6 prompts, 6 011 tokens in all,
// 5 412 -> 5 267 us a step; 4 of 1 500: 2 122 -> 2 023; one of 60: 1 018 -> 899.  (Launched on the step's own stream, with nothing waiting for it, 892 for 60 and
// 1 948: but what copies had left was there for any stream.)
constexpr int PLAN_SEQ = 128;
struct PlanSeqs {
  int start[PLAN_SEQ], slot[PLAN_SEQ], cu[PLAN_SEQ + 1];
};
__global__ __launch_bounds__(256) void step_plan_kernel(PlanSeqs a, int first, int capacity, int* __restrict__ cu, int* __restrict__ start,
                                                        int* __restrict__ slot, int* __restrict__ rows, int* __restrict__ seq,
                                                        int* __restrict__ keys) {
  const int i = blockIdx.y, b = first + i, st = a.start[i], lo = a.cu[i], n = a.cu[i + 1] - lo, row = a.slot[i] * capacity + st;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (b == 0) cu[0] = 0;
    cu[b + 1] = lo + n;
    start[b] = st;
    slot[b] = a.slot[i];
    if (keys) keys[b] = st + 1;
  }
  for (int t = blockIdx.x * 256 + threadIdx.x; t < n; t += 256 * gridDim.x) {
    rows[lo + t] = row + t;
    seq[lo + t] = b;
  }
}

}  // namespace

// A stream of the framework's own: those of torch's pool are handed out again, and one of them may be under capture in another thread when a step is planned
extern "C" int tv_step_plan_stream(void** stream) {
  TV_CHECK_ARG(stream, "step_plan_stream: null pointer");
  constexpr int MOST = 64;
  static std::mutex lock;
  static hipStream_t made[MOST];
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e == hipSuccess) {
    TV_CHECK_ARG(device >= 0 && device < MOST, "step_plan_stream: device %d", device);
    std::lock_guard<std::mutex> held(lock);
    if (!made[device]) e = hipStreamCreateWithFlags(&made[device], hipStreamNonBlocking);
    *stream = made[device];
  }
  if (e != hipSuccess) {
    tv_set_error("step_plan_stream: %s", hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  return TV_OK;
}

extern "C" int tv_step_plan(const int* starts, const int* slots, const int* counts, int sequences, int capacity, int* cu, int* start, int* slot,
                            int* rows, int* seq, int* keys, void* stream) {
  TV_CHECK_ARG(starts && slots && counts && cu && start && slot && rows && seq, "step_plan: null pointer");
  TV_CHECK_ARG(sequences > 0 && capacity > 0, "step_plan: %d sequences, capacity %d", sequences, capacity);
  int64_t total = 0;
  for (int b = 0; b < sequences; ++b) {
    TV_CHECK_ARG(starts[b] >= 0 && counts[b] > 0 && slots[b] >= 0 && (int64_t)starts[b] + counts[b] <= capacity,
                 "step_plan: sequence %d: %d tokens behind %d in slot %d of %d places", b, counts[b], starts[b], slots[b], capacity);
    total += counts[b];
    if (total > 0x3fffffff || ((int64_t)slots[b] + 1) * capacity > 0x7fffffff) TV_UNSUPPORTED("step_plan: rows beyond 32 bits");
  }
  int at = 0;
  for (int first = 0; first < sequences; first += PLAN_SEQ) {
    const int m = sequences - first < PLAN_SEQ ? sequences - first : PLAN_SEQ;
    PlanSeqs a;
    int most = 0;
    a.cu[0] = at;
    for (int i = 0; i < m; ++i) {
      a.start[i] = starts[first + i];
      a.slot[i] = slots[first + i];
      a.cu[i + 1] = at += counts[first + i];
      most = counts[first + i] > most ? counts[first + i] : most;
    }
    const int blocks = (most + 1023) / 1024;
    step_plan_kernel<<<dim3((unsigned)(blocks < 64 ? blocks : 64), (unsigned)m), 256, 0, (hipStream_t)stream>>>(a, first, capacity, cu, start, slot, rows,
                                                                                                              seq, keys);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      tv_set_error("step_plan: %s", hipGetErrorString(e));
      return TV_ERR_LAUNCH;
    }
  }
  return TV_OK;
}

extern "C" int tv_kv_append(const void* k, const void* v, void* k_cache, void* v_cache, const int64_t* pos, int batch, int64_t capacity, int row_bytes,
                            int64_t k_stride_b, int64_t v_stride_b, int64_t kc_stride_b, int64_t kc_stride_l, int64_t vc_stride_b,
                            int64_t vc_stride_l, void* stream) {
  TV_CHECK_ARG(k && v && k_cache && v_cache && pos, "kv_append: null pointer");
  TV_CHECK_ARG(batch > 0 && capacity > 0 && row_bytes > 0, "kv_append: bad sizes");
  if ((row_bytes | k_stride_b | v_stride_b | kc_stride_b | kc_stride_l | vc_stride_b | vc_stride_l | (int64_t)(uintptr_t)k | (int64_t)(uintptr_t)v |
       (int64_t)(uintptr_t)k_cache | (int64_t)(uintptr_t)v_cache) & 15)
    TV_UNSUPPORTED("kv_append: rows and strides (bytes) must be multiples of 16");
  kv_append_kernel<<<dim3((unsigned)batch, 2), 256, 0, (hipStream_t)stream>>>((const uint4*)k, (const uint4*)v, (uint4*)k_cache, (uint4*)v_cache, pos,
                                                                              capacity, row_bytes / 16, k_stride_b / 16, v_stride_b / 16,
                                                                              kc_stride_b / 16, kc_stride_l / 16, vc_stride_b / 16, vc_stride_l / 16);
  TV_LAUNCH_CHECK();
}

extern "C" int tv_count_up(int64_t* pos, int* lens, int n, void* stream) {
  TV_CHECK_ARG(pos && (lens || n == 0) && n >= 0, "count_up: bad arguments");
  count_up_kernel<<<1, 256, 0, (hipStream_t)stream>>>(pos, lens, n);
  TV_LAUNCH_CHECK();
}

extern "C" size_t tv_argmax_rows_workspace_bytes(int rows) { return rows > 0 ? (size_t)rows * ARG_BLOCKS * sizeof(Best) : 0; }

extern "C" int tv_argmax_rows(const float* x, int64_t* out, int rows, int n, int64_t stride, void* workspace, size_t workspace_bytes, void* stream) {
  return tv_argmax_rows_count(x, out, rows, n, stride, nullptr, nullptr, 0, workspace, workspace_bytes, stream);
}

extern "C" int tv_argmax_rows_count(const float* x, int64_t* out, int rows, int n, int64_t stride, int64_t* pos, int* lens, int nlens, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(nlens >= 0 && (lens || nlens == 0), "argmax_rows: %d counters", nlens);
  TV_CHECK_ARG(x && out && workspace, "argmax_rows: null pointer");
  TV_CHECK_ARG(rows > 0 && rows <= 65535 && n > 0 && stride >= 0, "argmax_rows: rows %d, %d elements", rows, n);
  if (n > (1 << 30)) TV_UNSUPPORTED("argmax_rows: %d elements a row, at most 2^30 (positions and the step behind the last share are 32-bit)", n);
  TV_CHECK_ARG(workspace_bytes >= tv_argmax_rows_workspace_bytes(rows) && ((uintptr_t)workspace & 7) == 0, "argmax_rows: workspace too small");
  const int wide = n % 4 == 0 && stride % 4 == 0 && ((uintptr_t)x & 15) == 0;
  argmax_part_kernel<<<dim3(ARG_BLOCKS, (unsigned)rows), 256, 0, (hipStream_t)stream>>>(x, (Best*)workspace, n, stride, wide);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    tv_set_error("argmax_rows: %s", hipGetErrorString(e));
    return TV_ERR_LAUNCH;
  }
  argmax_rows_kernel<<<(unsigned)rows, ARG_BLOCKS, 0, (hipStream_t)stream>>>((const Best*)workspace, out, pos, lens, nlens);
  TV_LAUNCH_CHECK();
}
