// The host side of the operators that short calls wait for, in C++: each function is one operator of kernels.py on operands that need no conversion - allocate the
// results, call the C entry point.  Anything else (a dtype or layout that kernels.py would convert, a tensor subclass, a wrapped or CPU tensor, an argument that it
// or the C entry refuses) returns None before anything is launched, and kernels.py goes its own way, errors included.  Where the C entry says that a launch failed,
// its kernels may be on their way all the same (the error can be an earlier call's): the operator is not run again, and raises what kernels.py would.
//
// A Python wrapper spends 5 - 10 us beside its 2.5 us launches on attribute calls, two more on the argument conversion of ctypes and 1.4 on every result; a short
// call's kernels are done before the next one is launched.  Host time of one call before -> now, us: norm 6.8 -> 3.9 (with a residual 8.4 -> 5.0), LayerNorm 7.1 -> 4.2,
// product of 33 - 256 rows 13.5 -> 7.4, small product 8.4 -> 4.6, attention 11.4 -> 5.6, a mixer's convolution, scan and gated norm together 41.5 -> 20.5.  Passes:
// 64 tokens of a mixer 44.5 -> 20.6 (its kernels), 1024 of a small fp32 one 42.3 -> 35.1, a prompt of 17 tokens 657 -> 545, of 100 945 -> 789, one video frame
// 2845 -> 2528, four packed prompts of 100 tokens 1215 -> 1045; from 700 tokens of a mixer and 300 of a prompt on the
// host is ahead either way.
#include <Python.h>
#include <dlfcn.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "timeviper_hip.h"

namespace {

#define TV_NATIVE_SYMBOLS(X)                                                                                                                              \
  X(tv_rmsnorm_fwd) X(tv_layernorm_fwd) X(tv_rmsnorm_gated_fwd) X(tv_causal_conv1d_xbc_fwd) X(tv_causal_conv1d_xbc_cb_fwd) X(tv_ssd_cb_bytes)              \
  X(tv_ssd_scan_workspace_bytes) X(tv_ssd_scan_cb_fwd) X(tv_flash_attn_fwd) X(tv_gemm_mid_fwd) X(tv_gemm_mid_workspace_bytes) X(tv_gemm_split_fwd)          \
  X(tv_gemm_mid_multi_fwd) X(tv_gemm_mid_multi_workspace_bytes) X(tv_gemm_small_add_fwd) X(tv_gemm_small_add_workspace_bytes)                                                                                        \
  X(tv_gemm_split_workspace_bytes) X(tv_gemm_split_add_fwd) X(tv_gemm_small_fwd) X(tv_gemm_rows_fwd) X(tv_residual_add_fwd)            \
  X(tv_token_side_fwd) X(tv_norm_shift_fwd) X(tv_gated_mul_fwd) X(tv_scatter_rows) X(tv_flash_attn_window_packed_fwd) X(tv_last_error)
struct Lib {
#define X(name) decltype(&::name) name = nullptr;
  TV_NATIVE_SYMBOLS(X)
#undef X
} lib;

typedef const at::Tensor* T;

struct Refused {};      // "kernels.py's way"
struct Failed {};       // a Python exception is set
PyObject* error = nullptr;      // the package's exception
inline void need(bool ok) { if (!ok) throw Refused{}; }

// an exact, dense-storage GPU tensor of the current device (None: nullptr, where allowed)
struct Operands {
  c10::DeviceIndex device = -1;
  T get(PyObject* o, bool optional = false) {
    if (o == Py_None) { need(optional); return nullptr; }
    need(THPVariable_CheckExact(o));
    T t = &THPVariable_Unpack(o);
    need(t->is_cuda() && t->layout() == at::kStrided && t->has_storage());
    if (device < 0) device = c10::hip::current_device();
    need(t->get_device() == device);
    return t;
  }
  void* stream() const { return (void*)c10::hip::getCurrentHIPStream(device).stream(); }
};
inline int dtype_of(T t) {
  switch (t->scalar_type()) {
    case at::kFloat: return TV_F32;
    case at::kBFloat16: return TV_BF16;
    case at::kHalf: return TV_F16;
    default: throw Refused{};
  }
}
inline bool bf16(T t) { return t->scalar_type() == at::kBFloat16; }
inline bool same_type(T a, T b) { return a->scalar_type() == b->scalar_type(); }
inline void* ptr(T t) { return t ? t->data_ptr() : nullptr; }
inline bool aligned(T t, uintptr_t n) { return t == nullptr || (uintptr_t)t->data_ptr() % n == 0; }
struct Unlocked {      // allocations and launches may wait for the GPU: other Python threads go on meanwhile, as beside torch's operators and ctypes
  PyThreadState* const state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
inline at::Tensor like(T t, at::IntArrayRef sizes) { Unlocked u; return at::empty(sizes, t->options()); }
inline at::Tensor like(T t, at::IntArrayRef sizes, at::ScalarType type) { Unlocked u; return at::empty(sizes, t->options().dtype(type)); }
inline int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  need(!(v == -1 && PyErr_Occurred()));
  return v;
}
inline double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  need(!(v == -1.0 && PyErr_Occurred()));
  return v;
}
inline bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  need(v >= 0);
  return v != 0;
}
template <typename F, typename... A>
void launch_named(const char* name, F f, A... args) {
  int status;
  { Unlocked u; status = f(args...); }
  need(status != TV_ERR_BAD_ARG && status != TV_ERR_UNSUPPORTED && status != TV_ERR_WORKSPACE);       // (nothing is launched: kernels.py calls again and says what was wrong)
  if (status != TV_OK) {
    PyErr_Format(error, "%s failed (status %d): %s", name, status, lib.tv_last_error());
    throw Failed{};
  }
}
#define launch(entry, ...) launch_named(#entry, lib.entry, __VA_ARGS__)
inline PyObject* wrap(at::Tensor&& t) { return THPVariable_Wrap(std::move(t)); }
template <typename... A>
PyObject* tuple(A*... items) {
  PyObject* const all[] = {items...};
  PyObject* r = PyTuple_New(sizeof...(items));
  for (size_t i = 0; i < sizeof...(items); ++i) {
    if (!r || !all[i]) { Py_XDECREF(r); return nullptr; }
    PyTuple_SET_ITEM(r, i, all[i]);
  }
  return r;
}
inline PyObject* again(PyObject* o) { Py_INCREF(o); return o; }

// ---- norms
// rms_norm(x, weight, eps, residual, return_sum)
PyObject* rms_norm(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), r = op.get(a[3], true);
  const bool sums = truth(a[4]);
  need(x->dim() > 0 && x->is_contiguous() && w->is_contiguous() && (w->scalar_type() == at::kFloat || same_type(w, x)));
  need(r == nullptr || (r->is_contiguous() && same_type(r, x) && r->sizes() == x->sizes()));
  const int64_t D = x->size(-1);
  need(D > 0 && w->numel() == D);
  at::Tensor y = like(x, x->sizes()), s;
  if (sums && r) s = like(x, x->sizes());
  launch(tv_rmsnorm_fwd, ptr(x), ptr(r), ptr(w), s.defined() ? s.data_ptr() : nullptr, y.data_ptr(), x->numel() / D, (int)D, D, r ? D : 0, s.defined() ? D : 0, D,
                            (float)real(a[2]), dtype_of(x), dtype_of(w), op.stream());
  if (!sums) return wrap(std::move(y));
  return tuple(wrap(std::move(y)), s.defined() ? wrap(std::move(s)) : again(a[0]));
}
// layer_norm(x, weight, bias, eps, return_sum, row_bias), no residual
PyObject* layer_norm(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), b = op.get(a[2], true), rb = op.get(a[5], true);
  need(x->dim() > 0 && x->is_contiguous() && same_type(w, x) && w->is_contiguous() && (b == nullptr || (same_type(b, x) && b->is_contiguous())));
  const int64_t D = x->size(-1);
  need(D > 0 && w->numel() == D && (b == nullptr || b->numel() == D) && (rb == nullptr || (rb->scalar_type() == at::kFloat && rb->is_contiguous() && rb->numel() == D)));
  const bool sums = truth(a[4]);
  at::Tensor y = like(x, x->sizes());
  launch(tv_layernorm_fwd, ptr(x), nullptr, ptr(w), ptr(b), (const float*)ptr(rb), nullptr, y.data_ptr(), x->numel() / D, (int)D, D, 0, 0, D, (float)real(a[3]), dtype_of(x),
                              op.stream());
  return sums ? tuple(wrap(std::move(y)), again(a[0])) : wrap(std::move(y));
}
// gated_norm(x, weight, z, eps, group_size)
PyObject* gated_norm(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), z = op.get(a[2], true);
  need(x->dim() > 0 && x->is_contiguous() && w->is_contiguous() && (w->scalar_type() == at::kFloat || same_type(w, x)));
  need(z == nullptr || (same_type(z, x) && z->dim() == 3 && z->sizes() == x->sizes() && z->stride(2) == 1 && (z->size(0) == 1 || z->stride(0) == z->size(1) * z->stride(1))));
  const int64_t D = x->size(-1), gs = a[4] == Py_None ? D : integer(a[4]);
  need(D > 0 && gs > 0 && gs <= D && w->numel() == D);
  at::Tensor y = like(x, x->sizes());
  launch(tv_rmsnorm_gated_fwd, ptr(x), ptr(z), ptr(w), y.data_ptr(), x->numel() / D, (int)D, (int)gs, D, z ? z->stride(1) : 0, D, (float)real(a[3]), dtype_of(x), dtype_of(w),
                                  op.stream());
  return wrap(std::move(y));
}

// ---- the mixer's operators
// conv_xbc(xBC, weight, bias, d_inner, ngroups, dstate, silu, return_cb)
PyObject* conv_xbc(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), b = op.get(a[2], true);
  const int64_t di = integer(a[3]), G = integer(a[4]), N = integer(a[5]);
  const bool silu = truth(a[6]), want_cb = truth(a[7]);
  need(x->dim() == 3 && di > 0 && G > 0 && N > 0 && x->size(2) == di + 2 * G * N && x->stride(2) == 1);
  const int64_t B = x->size(0), L = x->size(1), C = x->size(2), K = w->dim() ? w->size(-1) : 0;
  need(K > 0 && (w->dim() == 2 || w->dim() == 3) && w->numel() == C * K && w->size(0) == C && same_type(w, x) && w->is_contiguous());
  need(b == nullptr || (same_type(b, x) && b->is_contiguous() && b->numel() == C));
  at::Tensor yx = like(x, {B, L, di}), yb = like(x, {B, G, L, N}), yc = like(x, {B, G, L, N}), cb;
  if (want_cb && bf16(x) && N == 128 && L > 0) {
    cb = like(x, {(int64_t)(lib.tv_ssd_cb_bytes((int)B, (int)L, (int)G) / 2)});
    launch(tv_causal_conv1d_xbc_cb_fwd, ptr(x), ptr(w), ptr(b), nullptr, yx.data_ptr(), yb.data_ptr(), yc.data_ptr(), cb.data_ptr(), (int)B, (int)L, (int)di, (int)G, (int)N,
                                           (int)K, x->stride(0), x->stride(1), dtype_of(x), silu, op.stream());
  } else {
    launch(tv_causal_conv1d_xbc_fwd, ptr(x), ptr(w), ptr(b), nullptr, yx.data_ptr(), yb.data_ptr(), yc.data_ptr(), (int)B, (int)L, (int)di, (int)G, (int)N, (int)K,
                                        x->stride(0), x->stride(1), dtype_of(x), silu, op.stream());
  }
  PyObject *px = wrap(std::move(yx)), *pb = wrap(yb.transpose(1, 2)), *pc = wrap(yc.transpose(1, 2));
  if (!want_cb) return tuple(px, pb, pc);
  return tuple(px, pb, pc, cb.defined() ? wrap(std::move(cb)) : again(Py_None));
}
// rows of `inner` elements: the distances of batch entries and of rows
inline bool dense_rows(T t) {
  if (t->is_contiguous()) return true;
  int64_t expect = 1;
  for (int64_t d = t->dim() - 1; d > 1; --d) {
    if (t->stride(d) != expect) return false;
    expect *= t->size(d);
  }
  return t->stride(-1) == 1;
}
// scan(x, dt, A, B, C, D, dt_bias, initial_states, softplus, dt_min, dt_max, want_final, want_decay, group_map, cb)
PyObject* scan(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), dt = op.get(a[1]), A = op.get(a[2]), B = op.get(a[3]), C = op.get(a[4]), D = op.get(a[5], true), bias = op.get(a[6], true), init = op.get(a[7], true),
    cb = op.get(a[14], true);
  need(x->dim() == 4 && dt->dim() == 3 && B->dim() == 4 && C->dim() == 4 && same_type(dt, x) && same_type(B, x) && same_type(C, x));
  const int64_t b = x->size(0), L = x->size(1), H = x->size(2), P = x->size(3), G = B->size(2), N = B->size(3);
  need(dt->size(0) == b && dt->size(1) == L && dt->size(2) == H && B->size(0) == b && B->size(1) == L && C->sizes() == B->sizes());
  need(dense_rows(x) && dense_rows(dt) && B->stride(3) == 1 && C->stride(3) == 1);
  const auto f32 = [&](T t, int64_t n) { need(t == nullptr || (t->scalar_type() == at::kFloat && t->is_contiguous() && t->numel() == n)); };
  f32(A, H); f32(D, H); f32(bias, H); f32(init, b * H * P * N);
  need(D == nullptr || D->dim() == 1);
  need(cb == nullptr || (bf16(cb) && cb->is_contiguous() && (size_t)cb->numel() * 2 == lib.tv_ssd_cb_bytes((int)b, (int)L, (int)G)));
  const bool want_final = truth(a[11]), want_decay = truth(a[12]);
  at::Tensor y = like(x, {b, L, H, P}), fin, dec;
  if (want_final) fin = like(x, {b, H, P, N}, at::kFloat);
  if (want_decay) dec = like(x, {b, H}, at::kFloat);
  const size_t bytes = lib.tv_ssd_scan_workspace_bytes((int)b, (int)L, (int)H, (int)P, (int)G, (int)N, dtype_of(x));
  at::Tensor ws = like(x, {(int64_t)(bytes > 16 ? bytes : 16)}, at::kByte);
  launch(tv_ssd_scan_cb_fwd, ptr(x), ptr(dt), (const float*)ptr(A), ptr(B), ptr(C), ptr(cb), (const float*)ptr(D), (const float*)ptr(bias), (const float*)ptr(init), y.data_ptr(),
                                fin.defined() ? (float*)fin.data_ptr() : nullptr, dec.defined() ? (float*)dec.data_ptr() : nullptr, (int)b, (int)L, (int)H, (int)P, (int)G, (int)N,
                                x->stride(0), x->stride(1), dt->stride(0), dt->stride(1), B->stride(0), B->stride(1), B->stride(2), C->stride(0), C->stride(1), C->stride(2),
                                y.stride(0), y.stride(1), dtype_of(x), truth(a[8]), (float)real(a[9]), (float)real(a[10]), (int)integer(a[13]), ws.data_ptr(), bytes, op.stream());
  if (!want_final && !want_decay) return wrap(std::move(y));
  if (want_final && want_decay) return tuple(wrap(std::move(y)), wrap(std::move(fin)), wrap(std::move(dec)));
  return tuple(wrap(std::move(y)), wrap(std::move(want_final ? fin : dec)));
}

// ---- attention: flash(q, k, v, scale or None, causal, return_lse), more than one query row
PyObject* flash(PyObject* const* a) {
  Operands op;
  T q = op.get(a[0]), k = op.get(a[1]), v = op.get(a[2]);
  need(q->dim() == 4 && k->dim() == 4 && v->dim() == 4 && same_type(k, q) && same_type(v, q) && !(q->scalar_type() == at::kFloat));
  const int64_t B = q->size(0), Lq = q->size(1), H = q->size(2), D = q->size(3), Lk = k->size(1), G = k->size(2);
  need(Lq > 1 && B > 0 && D % 8 == 0 && D > 0 && k->size(0) == B && k->size(3) == D && v->sizes() == k->sizes());
  for (T t : {q, k, v}) need(t->stride(3) == 1 && t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0 && t->stride(2) % 8 == 0 && aligned(t, 16));
  const double scale = a[3] == Py_None ? 1.0 / std::sqrt((double)D) : real(a[3]);
  const bool want_lse = truth(a[5]);
  at::Tensor o = like(q, {B, Lq, H, D}), lse;
  if (want_lse) lse = like(q, {B, H, Lq}, at::kFloat);
  launch(tv_flash_attn_fwd, ptr(q), ptr(k), ptr(v), o.data_ptr(), want_lse ? lse.data_ptr() : nullptr, (int)B, (int)Lq, (int)Lk, (int)H, (int)G, (int)D, q->stride(0), q->stride(1),
                               q->stride(2), k->stride(0), k->stride(1), k->stride(2), v->stride(0), v->stride(1), v->stride(2), o.stride(0), o.stride(1), o.stride(2), (float)scale,
                               truth(a[4]), dtype_of(q), op.stream());
  return want_lse ? tuple(wrap(std::move(o)), wrap(std::move(lse))) : wrap(std::move(o));
}

// ---- products
struct Product {
  T x, w, b;
  int64_t M, N, K;
  at::Tensor y;
};
// x (..., K) dense, w (N, K) rows, bias of x's dtype (any_bias: or fp32), y (..., N)
void product(Operands& op, PyObject* const* a, Product& p, bool any_bias) {
  p.x = op.get(a[0]); p.w = op.get(a[1]); p.b = op.get(a[2], true);
  need(bf16(p.x) && bf16(p.w) && p.w->dim() == 2 && p.w->stride(1) == 1 && p.x->dim() > 0 && p.x->is_contiguous());
  p.N = p.w->size(0); p.K = p.w->size(1);
  need(p.K > 0 && p.N > 0 && p.x->size(-1) == p.K && p.x->numel() > 0);
  p.M = p.x->numel() / p.K;
  need(p.b == nullptr || ((bf16(p.b) || (any_bias && p.b->scalar_type() == at::kFloat)) && p.b->is_contiguous() && p.b->numel() == p.N));
  c10::SmallVector<int64_t, 5> sizes(p.x->sizes().begin(), p.x->sizes().end());
  sizes.back() = p.N;
  p.y = like(p.x, sizes);
}
// mid_linear(x, weight, bias, relu2)
PyObject* mid_linear(PyObject* const* a) {
  Operands op;
  Product p;
  product(op, a, p, false);
  need(p.K % 8 == 0 && p.K < (1 << 22) && aligned(p.x, 16) && aligned(p.b, 8));
  const size_t bytes = lib.tv_gemm_mid_workspace_bytes((int)p.M, (int)p.N, (int)p.K);
  at::Tensor ws;
  if (bytes) ws = like(p.x, {(int64_t)bytes}, at::kByte);
  launch(tv_gemm_mid_fwd, ptr(p.x), ptr(p.w), ptr(p.b), p.y.data_ptr(), (int)p.M, (int)p.N, (int)p.K, p.K, p.w->stride(0), p.N, truth(a[3]) ? TV_GEMM_ROWS_RELU2 : 0,
                             bytes ? ws.data_ptr() : nullptr, bytes, op.stream());
  return wrap(std::move(p.y));
}
// mid_linears(x, weight, weight, weight): the shapes are kernels.mid_linears_take's
PyObject* mid_linears(PyObject* const* a) {
  Operands op;
  const T x = op.get(a[0]);
  need(bf16(x) && x->dim() > 0 && x->is_contiguous() && aligned(x, 16));
  const int64_t K = x->size(-1), M = K > 0 ? x->numel() / K : 0;
  need(M >= 2 && M <= TV_GEMM_MID_MAX && K >= 4096 && K % 64 == 0 && K < (1 << 22));
  const void* W[3];
  void* Y[3];
  int N[3];
  int64_t ldw[3], ldy[3], all = 0;
  at::Tensor y[3];
  for (int i = 0; i < 3; ++i) {
    const T w = op.get(a[1 + i]);
    need(bf16(w) && w->dim() == 2 && w->size(1) == K && w->size(0) > 0 && w->size(0) % 4 == 0 && w->size(0) < (1 << 28) && w->stride(1) == 1 && w->stride(0) % 8 == 0 &&
         w->stride(0) >= K && w->stride(0) < (1 << 22) && aligned(w, 16));
    W[i] = ptr(w);
    N[i] = (int)w->size(0);
    ldw[i] = w->stride(0);
    ldy[i] = N[i];
    all += N[i];
  }
  need(all >= 4096);
  c10::SmallVector<int64_t, 5> sizes(x->sizes().begin(), x->sizes().end());
  for (int i = 0; i < 3; ++i) {
    sizes.back() = N[i];
    y[i] = like(x, sizes);
    Y[i] = y[i].data_ptr();
  }
  const size_t bytes = lib.tv_gemm_mid_multi_workspace_bytes((int)M, N, 3, (int)K);
  at::Tensor ws;
  if (bytes) ws = like(x, {(int64_t)bytes}, at::kByte);
  launch(tv_gemm_mid_multi_fwd, ptr(x), W, Y, N, 3, (int)M, (int)K, K, ldw, ldy, bytes ? ws.data_ptr() : nullptr, bytes, op.stream());
  return tuple(wrap(std::move(y[0])), wrap(std::move(y[1])), wrap(std::move(y[2])));
}
// split_linear(x, weight, bias, relu2, splits, full)
PyObject* split_linear(PyObject* const* a) {
  Operands op;
  Product p;
  product(op, a, p, true);
  const int splits = (int)integer(a[4]), full = (int)integer(a[5]);
  const size_t bytes = lib.tv_gemm_split_workspace_bytes(p.M, (int)p.N, splits, full);
  at::Tensor ws;
  if (bytes) ws = like(p.x, {(int64_t)bytes}, at::kByte);
  launch(tv_gemm_split_fwd, ptr(p.x), ptr(p.w), ptr(p.b), p.y.data_ptr(), p.M, (int)p.N, (int)p.K, p.K, p.w->stride(0), p.N, truth(a[3]) ? 3 : 0, p.b ? dtype_of(p.b) : TV_F32,
                               splits, full, bytes ? ws.data_ptr() : nullptr, bytes, op.stream());
  return wrap(std::move(p.y));
}
// rows_linear(x, weight, bias, epilogue): bf16 results, no convolution; the shapes are kernels.rows_take's
PyObject* rows_linear(PyObject* const* a) {
  Operands op;
  Product p;
  product(op, a, p, false);
  need(p.M >= 2 && p.M <= TV_GEMM_ROWS_MAX && p.K % 64 == 0 && p.K < (1 << 24) && p.w->stride(0) % 8 == 0 && p.w->stride(0) < (1 << 24) && aligned(p.w, 16) && aligned(p.x, 16));
  launch(tv_gemm_rows_fwd, ptr(p.x), ptr(p.w), ptr(p.b), p.y.data_ptr(), TV_BF16, (int)p.M, (int)p.N, (int)p.K, p.K, p.w->stride(0), p.N, (int)integer(a[3]), nullptr, nullptr,
                              nullptr, 0, 0, op.stream());
  return wrap(std::move(p.y));
}
// small_linear(x, weight, bias, epilogue, out or None, tile): x (rows, K)
PyObject* small_linear(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), b = op.get(a[2], true), out = op.get(a[4], true);
  const int epi = (int)integer(a[3]);
  need(bf16(x) && bf16(w) && x->dim() == 2 && w->dim() == 2 && x->size(1) == w->size(1) && x->stride(1) == 1 && w->stride(1) == 1);
  const int64_t N = epi == 5 ? w->size(0) / 2 : w->size(0);
  need(b == nullptr || ((bf16(b) || b->scalar_type() == at::kFloat) && b->is_contiguous() && b->numel() == w->size(0)));
  at::Tensor y;
  if (out == nullptr) {
    need(epi != 2);
    y = like(x, {x->size(0), N});
  } else {
    need(out->dim() == 2 && out->size(0) == x->size(0) && out->size(1) == N && bf16(out) && out->stride(1) == 1);
  }
  launch(tv_gemm_small_fwd, ptr(x), ptr(w), epi == 2 ? nullptr : ptr(b), out ? ptr(out) : y.data_ptr(), x->size(0), (int)N, (int)w->size(1), x->stride(0), w->stride(0),
                               out ? out->stride(0) : N, epi, b ? dtype_of(b) : TV_F32, (int)integer(a[5]), op.stream());
  return out ? again(a[4]) : wrap(std::move(y));
}

// ---- packed prompts of parallel layers
// residual_add(x, u)
PyObject* residual_add(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), u = op.get(a[1]);
  need(x->scalar_type() == at::kFloat && x->dim() == 2 && x->is_contiguous() && u->sizes() == x->sizes() && u->stride(1) == 1);
  at::Tensor xo = like(x, x->sizes()), h = like(u, x->sizes());
  launch(tv_residual_add_fwd, (const float*)ptr(x), ptr(u), (float*)xo.data_ptr(), h.data_ptr(), x->size(0), (int)x->size(1), u->stride(0), dtype_of(u), op.stream());
  return tuple(wrap(std::move(xo)), wrap(std::move(h)));
}
// split_add_linear(x, weight, residual, bias, splits)
PyObject* split_add_linear(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), r = op.get(a[2]), b = op.get(a[3], true);
  need(bf16(x) && bf16(w) && x->dim() == 2 && w->dim() == 2 && x->size(1) == w->size(1) && x->stride(1) == 1 && w->stride(1) == 1);
  const int64_t M = x->size(0), N = w->size(0);
  need(r->scalar_type() == at::kFloat && r->dim() == 2 && r->size(0) == M && r->size(1) == N && r->is_contiguous());
  need(b == nullptr || (bf16(b) && b->is_contiguous() && b->numel() == N));
  const int splits = (int)integer(a[4]);
  at::Tensor xo = like(r, r->sizes()), h = like(x, r->sizes()), ws;
  const size_t bytes = lib.tv_gemm_split_workspace_bytes(M, (int)N, splits, 0);
  if (bytes) ws = like(x, {(int64_t)bytes}, at::kByte);
  launch(tv_gemm_split_add_fwd, ptr(x), ptr(w), ptr(b), (const float*)ptr(r), (float*)xo.data_ptr(), h.data_ptr(), M, (int)N, (int)w->size(1), x->stride(0), w->stride(0), TV_BF16,
                                   splits, 0, bytes ? ws.data_ptr() : nullptr, bytes, op.stream());
  return tuple(wrap(std::move(xo)), wrap(std::move(h)));
}
// small_add_linear(x, weight, residual, bias, tile, splits)
PyObject* small_add_linear(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), w = op.get(a[1]), r = op.get(a[2]), b = op.get(a[3], true);
  need(bf16(x) && bf16(w) && x->dim() == 2 && w->dim() == 2 && x->size(1) == w->size(1) && x->stride(1) == 1 && w->stride(1) == 1);
  const int64_t M = x->size(0), N = w->size(0);
  need(M > 0 && N > 0 && r->scalar_type() == at::kFloat && r->dim() == 2 && r->size(0) == M && r->size(1) == N && r->is_contiguous());
  need(b == nullptr || (bf16(b) && b->is_contiguous() && b->numel() == N));
  const int tile = (int)integer(a[4]), splits = (int)integer(a[5]);
  const size_t bytes = lib.tv_gemm_small_add_workspace_bytes(M, (int)N, splits);
  need(bytes > 0);
  at::Tensor xo = like(r, r->sizes()), h = like(x, r->sizes()), ws = like(x, {(int64_t)bytes}, at::kByte);
  launch(tv_gemm_small_add_fwd, ptr(x), ptr(w), ptr(b), (const float*)ptr(r), (float*)xo.data_ptr(), h.data_ptr(), M, (int)N, (int)w->size(1), x->stride(0), w->stride(0), tile, splits,
                                   ws.data_ptr(), bytes, op.stream());
  return tuple(wrap(std::move(xo)), wrap(std::move(h)));
}
// token_side(h, ids, table, gate, proj)
PyObject* token_side(PyObject* const* a) {
  Operands op;
  T h = op.get(a[0]), ids = op.get(a[1]), table = op.get(a[2]), gate = op.get(a[3]), proj = op.get(a[4]);
  for (T t : {h, table, gate, proj}) need(bf16(t) && t->dim() == 2 && t->stride(1) == 1);
  const int64_t n = h->size(0), D = h->size(1), S = gate->size(0);
  need(gate->size(1) == D && proj->size(0) == D && proj->size(1) == S && table->size(1) == S && ids->scalar_type() == at::kLong && ids->numel() == n && ids->is_contiguous());
  at::Tensor y = like(h, {n, D});
  launch(tv_token_side_fwd, ptr(h), (const int64_t*)ptr(ids), ptr(table), ptr(gate), ptr(proj), y.data_ptr(), n, (int)D, (int)S, table->size(0), h->stride(0), table->stride(0),
                               gate->stride(0), proj->stride(0), D, op.stream());
  return wrap(std::move(y));
}

inline void int32s(T t, int64_t n) { need(t->scalar_type() == at::kInt && t->numel() >= n && t->is_contiguous()); }
// norm_shift(x, gain, eps, pending, pending_weight, shift, state, plan's seq, cu, start, slot, rows or None, largest slot, decode, need_h)
PyObject* norm_shift(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), g = op.get(a[1]), p = op.get(a[3], true), pw = op.get(a[4], true), sh = op.get(a[5], true), st = op.get(a[6], true);
  need(x->scalar_type() == at::kFloat && x->dim() == 2 && x->is_contiguous() && g->numel() == 1);
  if (!sh) st = nullptr;
  const int64_t n = x->size(0), D = x->size(1);
  const int type = dtype_of(g);
  need(p == nullptr || (pw && p->sizes() == x->sizes() && same_type(p, g) && p->stride(1) == 1 && same_type(pw, g) && pw->numel() == D && pw->is_contiguous()));
  T seq = nullptr, cu = nullptr, start = nullptr, slot = nullptr;
  if (sh) {
    seq = op.get(a[7]); cu = op.get(a[8]); start = op.get(a[9]); slot = op.get(a[10]);
    T rows = op.get(a[11]);
    need(st && same_type(sh, g) && sh->numel() == D && sh->is_contiguous() && rows->numel() == n);
    const int64_t B = slot->numel();
    int32s(seq, n); int32s(cu, B + 1); int32s(start, B); int32s(slot, B);
    need(st->scalar_type() == at::kFloat && st->dim() == 3 && st->size(1) == 2 && st->size(2) == D && st->stride(2) == 1 && st->stride(1) == D && integer(a[12]) < st->size(0));
  }
  at::Tensor xo, h, hs;
  if (p) xo = like(x, x->sizes());
  if (truth(a[14]) || !sh) h = like(g, x->sizes());
  if (sh) hs = like(g, x->sizes());
  launch(tv_norm_shift_fwd, (const float*)ptr(x), ptr(p), p ? ptr(pw) : nullptr, p ? (float*)xo.data_ptr() : nullptr, ptr(g), ptr(sh), (float*)ptr(st), (const int*)ptr(seq),
                               (const int*)ptr(cu), (const int*)ptr(start), (const int*)ptr(slot), h.defined() ? h.data_ptr() : nullptr, hs.defined() ? hs.data_ptr() : nullptr, n,
                               (int)D, p ? p->stride(0) : 0, st ? st->stride(0) : 0, (float)real(a[2]), truth(a[13]), type, op.stream());
  return tuple(p ? wrap(std::move(xo)) : again(a[0]), h.defined() ? wrap(std::move(h)) : again(Py_None), hs.defined() ? wrap(std::move(hs)) : again(Py_None));
}
// gated_mul(a, b, act, ids, out)
PyObject* gated_mul(PyObject* const* a) {
  Operands op;
  T x = op.get(a[0]), b = op.get(a[1]), ids = op.get(a[3], true), out = op.get(a[4], true);
  need(x->dim() == 2 && b->dim() == 2 && same_type(b, x) && b->size(1) == x->size(1) && x->stride(1) == 1 && b->stride(1) == 1);
  const int64_t n = x->size(0);
  need(ids ? ids->scalar_type() == at::kLong && ids->numel() == n && ids->is_contiguous() : b->size(0) == n);
  need(out == nullptr || (out->sizes() == x->sizes() && same_type(out, x) && out->stride(1) == 1));
  at::Tensor y;
  if (!out) y = like(x, x->sizes());
  launch(tv_gated_mul_fwd, ptr(x), ptr(b), (const int64_t*)ptr(ids), out ? ptr(out) : y.data_ptr(), n, (int)x->size(1), x->stride(0), b->stride(0), out ? out->stride(0) : x->size(1),
                              b->size(0), (int)integer(a[2]), dtype_of(x), op.stream());
  return out ? again(a[4]) : wrap(std::move(y));
}
// scatter_rows(src, rows, dst) -> True
PyObject* scatter_rows(PyObject* const* a) {
  Operands op;
  T src = op.get(a[0]), rows = op.get(a[1]), dst = op.get(a[2]);
  need(src->dim() == 2 && dst->dim() == 2 && same_type(src, dst) && src->size(1) == dst->size(1) && src->stride(1) == 1 && dst->stride(1) == 1);
  int32s(rows, src->size(0));
  launch(tv_scatter_rows, ptr(src), (const int*)ptr(rows), ptr(dst), src->size(0), (int)src->size(1), src->stride(0), dst->stride(0), dtype_of(src), op.stream());
  return again(Py_True);
}
// attention_window(q, cache, plan's counts, starts, slots, kv_heads, scale, window, keep_first, gate, out, plan's rows, seq, cu, start, slot)
PyObject* attention_window(PyObject* const* a) {
  Operands op;
  T q = op.get(a[0]), c = op.get(a[1]), g = op.get(a[9], true), out = op.get(a[10], true);
  need(bf16(q) && bf16(c) && q->dim() == 3 && c->dim() == 3 && c->is_contiguous() && PyTuple_Check(a[2]) && PyTuple_Check(a[3]) && PyTuple_Check(a[4]));
  const int64_t n = q->size(0), H = q->size(1), dk = q->size(2), G = integer(a[5]), cap = c->size(1), W = c->size(2);
  need(G > 0 && H > 0 && H % G == 0 && W % G == 0);
  const int64_t dv = W / G - dk;
  const Py_ssize_t B = PyTuple_GET_SIZE(a[2]);
  need(dk > 0 && dk <= 128 && dv > 0 && dv <= 128 && dk % 8 == 0 && dv % 8 == 0 && PyTuple_GET_SIZE(a[3]) == B && PyTuple_GET_SIZE(a[4]) == B);
  c10::SmallVector<int, 64> rows, lens_q, lens_k, slots;
  need(op.get(a[11])->numel() == n);
  int32s(op.get(a[12]), n); int32s(op.get(a[13]), B + 1); int32s(op.get(a[14]), B); int32s(op.get(a[15]), B);
  int64_t total = 0;
  for (Py_ssize_t i = 0; i < B; ++i) {
    const int64_t count = integer(PyTuple_GET_ITEM(a[2], i)), start = integer(PyTuple_GET_ITEM(a[3], i)), slot = integer(PyTuple_GET_ITEM(a[4], i));
    need(count >= 0 && start >= 0 && start + count <= cap && slot >= 0 && slot < c->size(0));
    rows.push_back((int)total); lens_q.push_back((int)count); lens_k.push_back((int)(start + count)); slots.push_back((int)slot);
    total += count;
  }
  need(total == n && n > 0 && real(a[6]) > 0);
  need(q->stride(2) == 1 && q->stride(0) % 8 == 0 && q->stride(1) % 8 == 0 && aligned(q, 16) && W % 8 == 0 && aligned(c, 16));
  for (T t : {g, out})
    need(t == nullptr || (bf16(t) && t->dim() == 3 && t->size(0) == n && t->size(1) == H && t->size(2) == dv && t->stride(2) == 1 && t->stride(0) % 4 == 0 && t->stride(1) % 4 == 0 &&
                          aligned(t, 8)));
  at::Tensor y;
  if (!out) y = like(q, {n, H, dv});
  char* const base = (char*)ptr(c);
  launch(tv_flash_attn_window_packed_fwd, ptr(q), base, base + G * dk * 2, out ? ptr(out) : y.data_ptr(), ptr(g), (int)integer(a[7]), (int)integer(a[8]), (int)dv, (int)B,
                                             rows.data(), lens_q.data(), lens_k.data(), slots.data(), (int)H, (int)G, (int)dk, q->stride(0), q->stride(1), cap * W, W, dk, cap * W, W, dv,
                                             out ? out->stride(0) : H * dv, out ? out->stride(1) : dv, g ? g->stride(0) : 0, g ? g->stride(1) : 0, (float)real(a[6]), TV_BF16,
                                             op.stream());
  return out ? again(a[10]) : wrap(std::move(y));
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != N || lib.tv_rmsnorm_fwd == nullptr) Py_RETURN_NONE;
  try {
    return F(args);
  } catch (const Failed&) {
    return nullptr;
  } catch (...) {              // (a C++ exception stays on this side)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// bind(path of the library that is loaded already, the exception for launches that fail)
PyObject* bind(PyObject*, PyObject* args) {
  const char* p;
  PyObject* e;
  if (!PyArg_ParseTuple(args, "sO", &p, &e)) return nullptr;
  void* h = dlopen(p, RTLD_NOW | RTLD_NOLOAD);
  if (!h) return PyErr_Format(PyExc_RuntimeError, "%s is not loaded", p);
  Lib l;
#define X(name)                                                                                    \
  if (!(l.name = (decltype(l.name))dlsym(h, #name))) {                                             \
    dlclose(h);                                                                                    \
    return PyErr_Format(PyExc_RuntimeError, "%s: no symbol %s", p, #name);                         \
  }
  TV_NATIVE_SYMBOLS(X)
#undef X
  lib = l;                     // (the handle is kept: the library stays mapped)
  Py_XDECREF(error);
  error = again(e);
  Py_RETURN_NONE;
}

#define ENTRY(name, n) {#name, (PyCFunction)(void*)(entry<name, n>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ENTRY(rms_norm, 5), ENTRY(layer_norm, 6), ENTRY(gated_norm, 5), ENTRY(conv_xbc, 8), ENTRY(scan, 15), ENTRY(flash, 6), ENTRY(mid_linear, 4), ENTRY(mid_linears, 4),
                         ENTRY(split_linear, 6), ENTRY(rows_linear, 4), ENTRY(small_linear, 6), ENTRY(residual_add, 2), ENTRY(split_add_linear, 5), ENTRY(small_add_linear, 6), ENTRY(token_side, 5), ENTRY(norm_shift, 15),
                         ENTRY(gated_mul, 5), ENTRY(scatter_rows, 3), ENTRY(attention_window, 16),
                         {"bind", (PyCFunction)bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tv_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tv_native() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_from", TV_NATIVE_ID) < 0) { Py_DECREF(m); return nullptr; }      // build.native_id() of the sources
  return m;
}
