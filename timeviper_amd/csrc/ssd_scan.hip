// S3 dispatcher: tv_ssd_scan_fwd picks an MFMA march kernel (bf16, d_state 128, MFMA-tileable head_dim, a
// workspace supplied: the head-per-wave march, else a slice march) or the generic fp32 path (chunk-parallel
// with a workspace and a small d_state, else the token recurrence).
#include <atomic>
#include "common.hpp"

int tv_ssd_generic_launch(const void* x, const void* dt, const void* A, const void* Bm,
                          const void* Cm, const void* D, const void* dt_bias,
                          const void* init_state, void* y, void* final_state, void* total_decay,
                          int batch, int seqlen, int nheads, int headdim, int ngroups, int dstate,
                          int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb,
                          int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg, int64_t ysb, int64_t ysl,
                          int dtype, int dt_softplus, float dt_min, float dt_max, int group_map,
                          hipStream_t st);

// ssd_slice.hip
bool tv_ssd_slice_supported(int seqlen, int nheads, int headdim, int ngroups, int dstate,
                            int dtype, int64_t xsl, int64_t bsl, int64_t bsg, int64_t csl, int64_t csg, int64_t ysl,
                            const void* x, const void* Bm, const void* Cm, const void* y, int wide);
size_t tv_ssd_slice_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int ngroups,
                                    int dstate, int wide);
int tv_ssd_slice_launch(const void* x, const void* dt, const void* A, const void* Bm,
                        const void* Cm, const void* D, const void* dt_bias,
                        const void* init_state, void* y, void* final_state, void* total_decay,
                        int batch, int seqlen, int nheads, int headdim, int ngroups, int dstate,
                        int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb,
                        int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg, int64_t ysb, int64_t ysl,
                        int dtype, int dt_softplus, float dt_min, float dt_max, int group_map,
                        void* workspace, size_t workspace_bytes, int wide, const void* cb_pre, hipStream_t st);

// ssd_chunked.hip: the generic path's chunk-parallel form (small d_state, any dtype)
bool tv_ssd_f32_supported(int headdim, int dstate, int64_t xsb, int64_t xsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg,
                          int64_t ysb, int64_t ysl, const void* x, const void* Bm, const void* Cm, const void* y, const void* init, const void* final_state);
int tv_ssd_f32_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* D, const void* dt_bias, const void* init_state,
                      void* y, void* final_state, void* total_decay, int batch, int seqlen, int nheads, int headdim, int ngroups, int64_t xsb, int64_t xsl,
                      int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg, int64_t ysb, int64_t ysl,
                      int dt_softplus, float dt_min, float dt_max, int group_map, bool fine, void* workspace, size_t workspace_bytes, hipStream_t st);
size_t tv_ssd_f32_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int dstate);
bool tv_ssd_chunked_supported(int seqlen, int headdim, int dstate);
size_t tv_ssd_chunked_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int dstate);
int tv_ssd_chunked_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm, const void* D,
                          const void* dt_bias, const void* init_state, void* y, void* final_state, void* total_decay,
                          int batch, int seqlen, int nheads, int headdim, int ngroups, int dstate, int64_t xsb, int64_t xsl,
                          int64_t dsb, int64_t dsl, int64_t bsb, int64_t bsl, int64_t bsg, int64_t csb, int64_t csl,
                          int64_t csg, int64_t ysb, int64_t ysl, int dtype, int dt_softplus, float dt_min, float dt_max,
                          int group_map, void* workspace, bool vector_only, int* ran, hipStream_t st);

// ssd_head.hip
bool tv_ssd_head_supported(int seqlen, int nheads, int headdim, int ngroups, int dstate, int dtype,
                           int64_t xsl, int64_t bsl, int64_t bsg, int64_t csl, int64_t csg, int64_t ysl,
                           const void* x, const void* Bm, const void* Cm, const void* y);
size_t tv_ssd_head_workspace_bytes(int batch, int seqlen, int nheads, int headdim, int ngroups, bool march_only);
int tv_ssd_head_launch(const void* x, const void* dt, const void* A, const void* Bm, const void* Cm,
                       const void* D, const void* dt_bias, const void* init_state, void* y,
                       void* final_state, void* total_decay, int batch, int seqlen, int nheads, int headdim,
                       int ngroups, int64_t xsb, int64_t xsl, int64_t dsb, int64_t dsl, int64_t bsb,
                       int64_t bsl, int64_t bsg, int64_t csb, int64_t csl, int64_t csg, int64_t ysb,
                       int64_t ysl, int dt_softplus, float dt_min, float dt_max, int group_map,
                       void* workspace, size_t workspace_bytes, const void* cb_pre, bool march_only, int* ran, hipStream_t st);

// 0 auto, 1 generic token recurrence (ssd_generic.hip: the definition), 3 slice march, two or more work-groups per head
// (ssd_slice.hip: the fallback for head dims that split into <= 40-column slices), 4 slice march, whole-head work-groups
// (head_dim 56 .. 80) x concurrent sequence segments + carried-in state correction (ssd_slice.hip + ssd_correct.hip),
// 6 head-per-wave march (ssd_head.hip: a wave owns a head, a work-group the heads of one B/C group, up to 16 sequence
// segments + correction; head_dim 32 / 64 / 80), 8 the generic path in chunk-parallel form (ssd_chunked.hip: small
// d_state, 2 .. 64 chunks) — what automatic selection takes where no march applies.
// Automatic selection has three more kernels, by its own rules and not to be forced, each of the family whose shapes it takes: 9 column slices (ssd_cols.hip) and
// 10 heads in segments (ssd_par.hip), both of family 6, 11 the matrix cores' form of 8 (ssd_f32.hip).  Forced, 6 is the march and 8 is ssd_chunked.hip.
// Removed as the slower ones: 2 (a chunk march; the number now means 3), 5 (a 12-wave whole-head layout; now
// means 4), 7 (a head march with two waves a SIMD; now means 6).
// process-wide override for tests / dev tools; atomic so that concurrent callers never race on it
static std::atomic<int> g_ssd_impl{0};
constexpr int F32_FROM = 48;          // tokens
static const int kAutoImpl = 6;   // head-per-wave march; falls back to 4, 3, the generic path

extern "C" void tv_ssd_scan_set_impl(int impl) { g_ssd_impl.store(impl, std::memory_order_relaxed); }
// which kernel family (0 .. 8 above), and which kernel (9 .. 11 as well), the most recent tv_ssd_scan_fwd / _cb_fwd of this process ran on; tests assert
// that a shape reached the kernel they mean to check
static std::atomic<int> g_ssd_last{0}, g_ssd_kernel{0};
extern "C" int tv_ssd_scan_last_impl(void) { return g_ssd_last.load(std::memory_order_relaxed); }
extern "C" int tv_ssd_scan_last_kernel(void) { return g_ssd_kernel.load(std::memory_order_relaxed); }
static void ran_on(int impl, int kernel) {
  g_ssd_last.store(impl, std::memory_order_relaxed);
  g_ssd_kernel.store(kernel, std::memory_order_relaxed);
}

extern "C" size_t tv_ssd_scan_workspace_bytes(int batch, int seqlen, int nheads, int headdim,
                                              int ngroups, int dstate, int dtype) {
  if (dtype != TV_BF16 || dstate != 128) {
    const size_t chunked = tv_ssd_chunked_workspace_bytes(batch, seqlen, nheads, headdim, dstate);
    const size_t f32 = dtype == TV_F32 ? tv_ssd_f32_workspace_bytes(batch, seqlen, nheads, headdim, dstate) : 0;
    const size_t m = chunked > f32 ? chunked : f32;
    // (one launch of ssd_f32.hip needs none, but a caller that gives none asks for the recurrence)
    return m == 0 && dtype == TV_F32 && dstate == 16 && seqlen > 64 ? 256 : (m + 255) / 256 * 256;
  }
  const size_t narrow = tv_ssd_slice_workspace_bytes(batch, seqlen, nheads, headdim, ngroups, dstate, 0);
  const size_t wide = tv_ssd_slice_workspace_bytes(batch, seqlen, nheads, headdim, ngroups, dstate, 1);
  const int forced = g_ssd_impl.load(std::memory_order_relaxed);
  const size_t head = tv_ssd_head_workspace_bytes(batch, seqlen, nheads, headdim, ngroups, forced == 6 || forced == 7);
  size_t m = narrow > wide ? narrow : wide;             // any variant may be selected (tv_ssd_scan_set_impl)
  return ((m > head ? m : head) + 255) / 256 * 256;
}

static int scan_impl(const void* x, const void* dt, const void* A, const void* Bm,
                     const void* Cm, const void* D, const void* dt_bias,
                     const void* init_state, void* y, void* final_state,
                     void* total_decay, int batch, int seqlen, int nheads, int headdim,
                     int ngroups, int dstate, int64_t x_stride_b, int64_t x_stride_l,
                     int64_t dt_stride_b, int64_t dt_stride_l, int64_t b_stride_b,
                     int64_t b_stride_l, int64_t b_stride_g, int64_t c_stride_b,
                     int64_t c_stride_l, int64_t c_stride_g, int64_t y_stride_b,
                     int64_t y_stride_l, int dtype, int dt_softplus,
                     float dt_min, float dt_max, int group_map, const void* cb, void* workspace,
                     size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(A && (seqlen == 0 || (x && dt && Bm && Cm && y)), "ssd_scan: null pointer");   // empty tensors have no storage
  TV_CHECK_ARG(batch > 0 && seqlen >= 0 && nheads > 0 && headdim > 0 && ngroups > 0 &&
                   dstate > 0 && nheads % ngroups == 0,
               "ssd_scan: bad sizes (B %d L %d H %d P %d G %d N %d)", batch, seqlen, nheads,
               headdim, ngroups, dstate);
  TV_CHECK_ARG(dtype == TV_F32 || dtype == TV_BF16 || dtype == TV_F16, "ssd_scan: dtype %d", dtype);
  hipStream_t st = (hipStream_t)stream;
  if (seqlen == 0) {
    // empty sequence: the state passes through unchanged
    if (final_state) {
      const size_t bytes = (size_t)batch * nheads * headdim * dstate * sizeof(float);
      if (init_state) (void)hipMemcpyAsync(final_state, init_state, bytes, hipMemcpyDeviceToDevice, st);
      else (void)hipMemsetAsync(final_state, 0, bytes, st);
    }
    if (total_decay) (void)hipMemsetAsync(total_decay, 0, (size_t)batch * nheads * sizeof(float), st);
    return TV_OK;
  }
  int forced = g_ssd_impl.load(std::memory_order_relaxed);   // one read per call
  if (forced == 2) forced = 3;          // removed kernels: the numbers select their successors
  if (forced == 5) forced = 4;
  if (forced == 7) forced = 6;
  const bool mfma_ok = forced != 1 && forced != 8 && workspace && dt_stride_l % 2 == 0 && dt_stride_b % 2 == 0 &&
                       (((uintptr_t)dt) & 3) == 0;
  const int impl = forced ? forced : kAutoImpl;
  if (mfma_ok && impl == 6 &&
      tv_ssd_head_supported(seqlen, nheads, headdim, ngroups, dstate, dtype, x_stride_l, b_stride_l, b_stride_g,
                            c_stride_l, c_stride_g, y_stride_l, x, Bm, Cm, y)) {
    // the head-per-wave march takes every chunk itself (floating, reset and standard steps in the one kernel)
    int ran = 6;
    const int rc = tv_ssd_head_launch(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state, total_decay, batch, seqlen,
                              nheads, headdim, ngroups, x_stride_b, x_stride_l, dt_stride_b, dt_stride_l, b_stride_b,
                              b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l,
                              dt_softplus, dt_min, dt_max, group_map, workspace, workspace_bytes, cb, forced == 6, &ran, st);
    ran_on(6, ran);
    return rc;
  }
  for (int wide = 1; wide >= 0; --wide) {       // impl 4 (and 6 where it does not apply): whole-head work-groups first, then slices of a head
    if (wide == 1 && impl != 4 && impl != 6) continue;
    if (mfma_ok && impl >= 3 &&
        tv_ssd_slice_supported(seqlen, nheads, headdim, ngroups, dstate, dtype, x_stride_l, b_stride_l,
                               b_stride_g, c_stride_l, c_stride_g, y_stride_l, x, Bm, Cm, y, wide)) {
      ran_on(wide == 1 ? 4 : 3, wide == 1 ? 4 : 3);
      return tv_ssd_slice_launch(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state,
                                 total_decay, batch, seqlen, nheads, headdim, ngroups, dstate,
                                 x_stride_b, x_stride_l, dt_stride_b, dt_stride_l, b_stride_b,
                                 b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, dtype,
                                 dt_softplus, dt_min, dt_max, group_map, workspace, workspace_bytes,
                                 wide, cb, st);
    }
  }
  if (forced >= 3 && forced != 8)
    TV_UNSUPPORTED("ssd_scan: MFMA march kernel forced but shape / dtype / alignment unsupported or no workspace given");
  if ((forced == 0 || forced == 8) && workspace && tv_ssd_chunked_supported(seqlen, headdim, dstate) &&
      workspace_bytes >= tv_ssd_chunked_workspace_bytes(batch, seqlen, nheads, headdim, dstate)) {
    int ran = 8;
    const int rc = tv_ssd_chunked_launch(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state, total_decay, batch, seqlen,
                                 nheads, headdim, ngroups, dstate, x_stride_b, x_stride_l, dt_stride_b, dt_stride_l,
                                 b_stride_b, b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b,
                                 y_stride_l, dtype, dt_softplus, dt_min, dt_max, group_map, workspace, forced == 8, &ran, st);
    ran_on(8, ran);
    return rc;
  }
  // Lengths that ssd_chunked.hip leaves out (up to 64 tokens, more than 4 096), on the matrix cores where their rows allow it.  us, token by token | here, 32 heads x 64: 48 tokens
  // 17.7 | 8.7, 64: 22 | 8.8, 8 192: 2 690 | 100; 128 x 128, 64: 28 | 9.8; 24: 10.2 | 7.4, left to the recurrence, whose error was the smaller one by some per cent when
  // the line was drawn
  if (forced == 0 && dtype == TV_F32 && workspace && (uintptr_t)workspace % 16 == 0 && seqlen >= F32_FROM &&
      tv_ssd_f32_supported(headdim, dstate, x_stride_b, x_stride_l, b_stride_b, b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, x,
                           Bm, Cm, y, init_state, final_state)) {
    ran_on(8, 11);
    return tv_ssd_f32_launch(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state, total_decay, batch, seqlen, nheads, headdim, ngroups, x_stride_b, x_stride_l,
                             dt_stride_b, dt_stride_l, b_stride_b, b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, dt_softplus, dt_min,
                             dt_max, group_map, true, workspace, workspace_bytes, st);
  }
  if (forced == 8) TV_UNSUPPORTED("ssd_scan: chunk-parallel generic kernel forced but shape unsupported");
  ran_on(1, 1);
  return tv_ssd_generic_launch(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state,
                               total_decay, batch, seqlen, nheads, headdim, ngroups, dstate,
                               x_stride_b, x_stride_l, dt_stride_b, dt_stride_l, b_stride_b,
                               b_stride_l, b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, dtype,
                               dt_softplus, dt_min, dt_max, group_map, st);
}

extern "C" int tv_ssd_scan_fwd(const void* x, const void* dt, const void* A, const void* Bm,
                               const void* Cm, const void* D, const void* dt_bias,
                               const void* init_state, void* y, void* final_state,
                               void* total_decay, int batch, int seqlen, int nheads, int headdim,
                               int ngroups, int dstate, int64_t x_stride_b, int64_t x_stride_l,
                               int64_t dt_stride_b, int64_t dt_stride_l, int64_t b_stride_b,
                               int64_t b_stride_l, int64_t b_stride_g, int64_t c_stride_b,
                               int64_t c_stride_l, int64_t c_stride_g, int64_t y_stride_b,
                               int64_t y_stride_l, int dtype, int dt_softplus,
                               float dt_min, float dt_max, int group_map, void* workspace,
                               size_t workspace_bytes, void* stream) {
  return scan_impl(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state, total_decay, batch, seqlen, nheads,
                   headdim, ngroups, dstate, x_stride_b, x_stride_l, dt_stride_b, dt_stride_l, b_stride_b, b_stride_l,
                   b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, dtype, dt_softplus, dt_min,
                   dt_max, group_map, nullptr, workspace, workspace_bytes, stream);
}

// The same scan with the causal C.B^T fragments of every (chunk, group) supplied by the caller — the `cb` output of
// tv_causal_conv1d_xbc_cb_fwd on the same B / C (tv_ssd_cb_bytes() bytes) — instead of recomputed by a pre-pass
// that reads B and C back.  Kernels that do not use the fragments (fp32, other d_state) ignore them.
extern "C" int tv_ssd_scan_cb_fwd(const void* x, const void* dt, const void* A, const void* Bm,
                                  const void* Cm, const void* cb, const void* D, const void* dt_bias,
                                  const void* init_state, void* y, void* final_state,
                                  void* total_decay, int batch, int seqlen, int nheads, int headdim,
                                  int ngroups, int dstate, int64_t x_stride_b, int64_t x_stride_l,
                                  int64_t dt_stride_b, int64_t dt_stride_l, int64_t b_stride_b,
                                  int64_t b_stride_l, int64_t b_stride_g, int64_t c_stride_b,
                                  int64_t c_stride_l, int64_t c_stride_g, int64_t y_stride_b,
                                  int64_t y_stride_l, int dtype, int dt_softplus,
                                  float dt_min, float dt_max, int group_map, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  TV_CHECK_ARG(cb == nullptr || (((uintptr_t)cb) & 15) == 0, "ssd_scan_cb: C.B^T buffer must be 16-byte aligned");
  return scan_impl(x, dt, A, Bm, Cm, D, dt_bias, init_state, y, final_state, total_decay, batch, seqlen, nheads,
                   headdim, ngroups, dstate, x_stride_b, x_stride_l, dt_stride_b, dt_stride_l, b_stride_b, b_stride_l,
                   b_stride_g, c_stride_b, c_stride_l, c_stride_g, y_stride_b, y_stride_l, dtype, dt_softplus, dt_min,
                   dt_max, group_map, cb, workspace, workspace_bytes, stream);
}
