"""The operators' native host side: the same kernels on the same operands, so the same bits as the way through Python, over the forms that both take; what it does not take."""
import ctypes
import dataclasses
import re
import subprocess
import threading

import pytest
import torch

from timeviper_amd import _capi, build
from timeviper_amd import kernels as ops
from timeviper_amd._native import ops as native

DEV = "cuda"
BF, F32, F16 = torch.bfloat16, torch.float32, torch.float16
NAMES = ("rms_norm", "layer_norm", "gated_norm", "conv_xbc", "scan", "flash", "mid_linear", "split_linear", "rows_linear", "small_linear", "residual_add", "split_add_linear",
         "token_side", "norm_shift", "gated_mul", "scatter_rows", "attention_window")


class Asked:
    """The native operators (or none of them), with a count of the calls that they took"""
    def __init__(self, on):
        self.on, self.took = on, 0

    def __getattr__(self, name):
        def call(*a):
            r = getattr(native, name)(*a) if self.on else None
            self.took += r is not None
            return r
        return call


def r(*s, dtype=BF, seed=0):
    return torch.randn(s, generator=torch.Generator(device=DEV).manual_seed(seed + sum(s)), device=DEV).to(dtype)


class Own(torch.Tensor):
    pass


def plan(counts, starts, slots, cap):
    from timeviper_amd.model.llm.cache import StepPlan
    i = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    cu = [sum(counts[:j]) for j in range(len(counts) + 1)]
    return StepPlan(slots=tuple(slots), counts=tuple(counts), starts=tuple(starts), cu=i(cu), start=i(starts), slot=i(slots),
                    rows=i([s * cap + a + j for s, a, n in zip(slots, starts, counts) for j in range(n)]), seq=i([b for b, n in enumerate(counts) for _ in range(n)]), keys=None, moving=None,
                    decode=False)


def norms(t):
    for x, res in ((r(7, 96, dtype=t), None), (r(2, 3, 4096, dtype=t), r(2, 3, 4096, dtype=t, seed=1)), (r(5, 64, dtype=t), r(5, 64, dtype=t, seed=2))):
        D = x.shape[-1]
        for w in {t: r(D, dtype=t), F32: r(D, dtype=F32)}.values():
            for sums in (False, True):
                yield lambda: ops.rms_norm(x, w, 1e-5, res, sums), 1
        for b in (None, r(D, dtype=t, seed=3)):
            for rb in (None, r(D, dtype=F32, seed=4)):
                yield lambda: ops.layer_norm(x, r(D, dtype=t), b, 1e-6, None, True, rb), 1
    z = r(2, 9, 704, dtype=t)                                                            # gates: columns of a wider projection
    for z_, group in ((None, 64), (z[..., 64:320], 64), (z[..., :256].contiguous(), None)):
        yield lambda: ops.rmsnorm_fn(r(2, 9, 256, dtype=t), r(256, dtype=F32), None, z_, 1e-5, group, norm_before_gate=False), 1
    yield lambda: ops.rms_norm(r(6, 96, dtype=t)[::2], r(96, dtype=t), 1e-5), 0           # a copy is needed
    yield lambda: ops.rms_norm(r(6, 96, dtype=t).as_subclass(Own), r(96, dtype=t), 1e-5), 0


def mixer(t):
    for B, L, cols in ((1, 1, 0), (2, 63, 40), (1, 300, 8)):
        H, P, G, N = 16, 64, 2, 128
        di = H * P
        wide = r(B, L, cols + di + 2 * G * N + H, dtype=t)
        xBC, dt = wide[..., cols:cols + di + 2 * G * N], wide[..., cols + di + 2 * G * N:]
        w, b = r(di + 2 * G * N, 1, 4, dtype=t), r(di + 2 * G * N, dtype=t)
        A, D, bias = -torch.rand(H, device=DEV) - .1, r(H, dtype=F32), r(H, dtype=F32)
        for cb in (False, True):
            yield lambda: ops.causal_conv1d_xbc(xBC, w.squeeze(1), b if cb else None, di, G, N, return_cb=cb), 1
        x, Bm, Cm = ops.causal_conv1d_xbc(xBC, w.squeeze(1), b, di, G, N)[:3]
        for init in (None, r(B, H, P, N, dtype=F32)):
            for final in (False, True):
                yield lambda: ops.mamba_chunk_scan_combined(x.view(B, L, H, P), dt, A, Bm, Cm, chunk_size=256, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=final), 1


def attention(t):
    for D, Lq, Lk in ((128, 5, 5), (72, 130, 130), (64, 33, 100)):
        wide = r(2, max(Lq, Lk), 8 * D, dtype=t)
        q, k, v = wide[:, :Lq, :4 * D].unflatten(2, (4, D)), wide[:, :Lk, 4 * D:6 * D].unflatten(2, (2, D)), wide[:, :Lk, 6 * D:].unflatten(2, (2, D))
        for causal in (False, True):
            for scale in (None, .3):
                yield lambda: ops.flash_attn_func(q, k, v, softmax_scale=scale, causal=causal, return_lse=causal), 1
    yield lambda: ops.flash_attn_func(r(2, 9, 4, 128, dtype=t)[..., ::2], r(2, 9, 2, 64, dtype=t), r(2, 9, 2, 64, dtype=t)), 0       # a copy is needed


def products(t):
    for M in (33, 100, 256):
        wide = r(640, 520)
        for w in (wide[:, :512], wide[:, :512].contiguous()):
            for b in (None, r(640)):
                yield lambda: ops.mid_linear(r(M, 512), w, b, relu2=b is None), 1
                yield lambda: ops.split_linear(r(M, 512), w, b, splits=2), 1
                yield lambda: ops.small_linear(r(M, 512), w, b, 1 if b is None else 0), 1
                yield lambda: ops.split_add_linear(r(M, 512), w, r(M, 640, dtype=F32), b, splits=2), 1
    for M in (2, 17, 32):
        yield lambda: ops.rows_linear(r(1, M, 512), r(640, 512), r(640) if M == 2 else None, relu2=M == 17), 1


def packed(t):
    dk, G, H, cap = 64, 2, 6, 200
    cache, p = r(3, cap, G * 2 * dk), plan([5, 1, 120], [0, 30, 80], [2, 0, 1], cap)
    T, D = 126, 96
    wide = r(T, 2 * H * dk)
    q, gate = wide[:, :H * dk].unflatten(1, (H, dk)), wide[:, H * dk:].unflatten(1, (H, dk))
    for g in (None, gate):
        for window in (7, 1 << 30):
            yield lambda: ops.attention_window(q, cache, p, G, .125, window=window, keep_first=4, gate=g), 1
    yield lambda: ops.attention_window(q, cache, p, G, .125, gate=gate, out=torch.empty(T, H, dk + 8, dtype=BF, device=DEV)[..., :dk]), 1
    x, y = r(T, D, dtype=F32), r(T, 2 * D)[:, D:]
    for pending in (None, y):
        yield lambda: ops.norm_shift(x, r(1), 1e-5, pending, None if pending is None else r(D)), 1
        state = r(3, 5, 2, D, dtype=F32)
        yield lambda: (ops.norm_shift(x, r(1), 1e-5, pending, None if pending is None else r(D), r(D), (s := state.clone())[:, 3], p, need_h=pending is None), s), 1
    yield lambda: ops.residual_add(x, y), 1
    ids = torch.arange(T, device=DEV).flip(0)
    for i, b in ((None, r(T, D, seed=5)), (ids, r(T, D, seed=6))):
        for act in (0, 1):
            yield lambda: ops.gated_mul(y, b, act, i), 1
    yield lambda: ops.gated_mul(y, r(T, D), 0, None, torch.empty(T, 2 * D, dtype=BF, device=DEV)[:, :D]), 1
    def scatter():
        dst = torch.zeros(3 * cap, D, dtype=BF, device=DEV)
        ops.scatter_rows(y, p.rows, dst)
        return dst
    yield scatter, 1


def products_more(t):
    """epilogues, rows to write to, splits behind whole tiles, the token side"""
    for M in (33, 200):
        x, w, wide = r(M, 512), r(640, 512), r(M, 700, seed=9)
        for tile in range(4):
            for b in (None, r(640), r(640, dtype=F32)):
                for epilogue in (ops.GEMM_BIAS, ops.GEMM_BIAS_GELU, ops.GEMM_GLU)[:3 if b is not None and b.dtype == t else 2]:       # (the gate: a bf16 bias)
                    yield lambda: ops.small_linear(x, w, b, epilogue, tile=tile), 1
                yield lambda: ops.small_linear(x, w, b, out=torch.empty(M, 704, dtype=BF, device=DEV)[:, 8:648], tile=tile), 1
                yield lambda: (ops.small_linear(x, w, b, ops.GEMM_ACCUM, (o := r(M, 704, seed=8))[:, 8:648], tile), o), 1
        for b in (None, r(640), r(640, dtype=F32)):
            yield lambda: ops.split_linear(x, w, b, True, 1), 1
    for b in (None, r(1024)):
        yield lambda: ops.split_linear(r(3, 200, 1024), r(1024, 1024), b, b is None, 3, 5), 1
        yield lambda: ops.split_linear(r(600, 1024), r(1024, 1024), b, False, 4, 8), 1
    for T, D in ((5, 64), (130, 256)):
        table, ids = r(50, 3, 128)[:, 1], torch.arange(T, device=DEV) * 7 % 50
        yield lambda: ops.token_side(r(T, 2 * D)[:, D:], ids, table, r(128, D + 8)[:, :D], r(D, 136)[:, 8:]), 1


def mixer_more(t):
    """all that a scan takes beside its operands, the convolution's C.B^T, the state sizes that go elsewhere"""
    for B, L, P, N, G in ((1, 300, 64, 128, 2), (2, 70, 80, 128, 8), (1, 64, 64, 16, 2), (2, 4100, 32, 16, 1)):
        H = 16
        di = H * P
        wide, w = r(B, L, 8 + di + 2 * G * N + H, dtype=t), r(di + 2 * G * N, 4, dtype=t)
        dt = wide[..., 8 + di + 2 * G * N:]
        A, D, bias, init = -torch.rand(H, device=DEV) - .1, r(H, dtype=F32), r(H, dtype=F32), r(B, H, P, N, dtype=F32)
        x, Bm, Cm, cb = ops.causal_conv1d_xbc(wide[..., 8:8 + di + 2 * G * N], w, None, di, G, N, return_cb=True)
        x = x.view(B, L, H, P)
        yield lambda: ops.causal_conv1d_xbc(wide[..., 8:8 + di + 2 * G * N], w, None, di, G, N, activation=None, return_cb=True), 1
        for c in {None, cb}:
            for final in (False, True):
                yield lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=final, return_total_decay=True, cb=c), 1
                yield lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, dt_bias=bias, dt_softplus=True, return_final_states=final, cb=c), 1
        yield lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_softplus=True, dt_limit=(.2, .5), return_total_decay=True), 1
        yield lambda: ops.mamba_chunk_scan_combined(x, dt.abs(), A, Bm, Cm, D=D, group_map="tile", return_final_states=True), 1


def packed_more(t):
    """a decoded token of every sequence: the state's other route"""
    B, D = 5, 96
    p = dataclasses.replace(plan([1] * B, [0, 3, 8, 1, 2], [4, 0, 1, 3, 2], 20), decode=True)
    x, y = r(B, D, dtype=F32), r(B, 2 * D)[:, D:]
    for pending in (None, y):
        for need in (False, True):
            state = r(5, 3, 2, D, dtype=F32)
            yield lambda: (ops.norm_shift(x, r(1), 1e-5, pending, None if pending is None else r(D), r(D), (s := state.clone())[:, 1], p, need_h=need), s), 1


def flat(v):
    return [t for u in v for t in flat(u)] if isinstance(v, (tuple, list)) else [v]


@pytest.mark.gpu
@pytest.mark.parametrize("forms,dtype", [(norms, BF), (norms, F32), (norms, F16), (mixer, BF), (mixer, F32), (attention, BF), (attention, F16), (products, BF), (packed, BF),
                                         (products_more, BF), (mixer_more, BF), (mixer_more, F32), (mixer_more, F16), (packed_more, BF)])
def test_same_bits(forms, dtype, monkeypatch):
    for call, taken in forms(dtype):
        got = []
        for on in (True, False):
            asked = Asked(on)
            monkeypatch.setattr(ops, "_n", asked)
            got.append(flat(call()))
            assert asked.took == (taken if on else 0)
        monkeypatch.setattr(ops, "_n", native)
        assert len(got[0]) == len(got[1])
        for a, b in zip(*got):
            if not isinstance(a, torch.Tensor):
                assert a is b is None
                continue
            assert type(a) is type(b) and a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
            bits = lambda t: t.contiguous().view(torch.uint8)
            assert torch.equal(bits(a), bits(b))


@pytest.mark.gpu
@pytest.mark.parametrize("call", [
    lambda: ops.flash_attn_func(r(2, 9, 4, 68)[..., :64], r(2, 9, 2, 64), r(2, 9, 2, 64)), lambda: ops.rms_norm(r(3, 64), torch.ones(64), 1e-5), lambda: ops.flash_attn_func(r(1, 4, 3, 64), r(1, 4, 2, 64), r(1, 4, 2, 64)),
    lambda: ops.residual_add(r(3, 64), r(3, 64)), lambda: ops.gated_mul(r(3, 64), r(4, 64), 0), lambda: ops.mid_linear(r(300, 512), r(640, 512)),
    lambda: ops.attention_window(r(4, 2, 64), r(1, 3, 256), plan([4], [0], [0], 3), 2, .1), lambda: ops.scatter_rows(r(4, 64), torch.zeros(3, dtype=torch.int32, device=DEV), r(9, 64))])
def test_refused_as_before(call, monkeypatch):
    told = []
    for on in (True, False):
        monkeypatch.setattr(ops, "_n", Asked(on))
        with pytest.raises(Exception) as e:
            call()
        told.append((type(e.value), str(e.value)))
    assert told[0] == told[1]


@pytest.fixture
def failing(tmp_path):
    """The native operators on a library whose every entry counts its calls and says that a launch failed"""
    entries = sorted(set(re.findall(r"X\((tv_\w+)\)", build.NATIVE_SRC.read_text())) - {"tv_last_error"})
    source, stub = tmp_path / "stub.c", tmp_path / "stub.so"
    source.write_text("int calls;\nconst char* tv_last_error(void) { return \"an earlier call's\"; }\n" +
                      "".join(f"{'unsigned long' if 'bytes' in e else 'int'} {e}(void) {{ {'return 0' if 'bytes' in e else '++calls; return -4'}; }}\n" for e in entries))
    subprocess.run(["gcc", "-shared", "-fPIC", str(source), "-o", str(stub)], check=True)
    lib = ctypes.CDLL(str(stub))
    native.rms_norm                                                                      # (loaded)
    native.bind(str(stub), ops.TimeViperHipError)
    yield ctypes.c_int.in_dll(lib, "calls")
    native.bind(str(_capi.lib_path()), ops.TimeViperHipError)


@pytest.mark.gpu
def test_a_failed_launch_raises_and_is_not_run_again(failing):
    """The kernel may be on its way (the error can be an earlier call's): an operator that changes its operands must not run twice."""
    x, w, out = r(40, 512), r(640, 512), r(40, 640)
    p, state = plan([4], [2], [0], 8), r(1, 2, 96, dtype=F32)
    before, state0 = out.clone(), state.clone()
    for n, (call, entry) in enumerate(((lambda: ops.small_linear(x, w, None, ops.GEMM_ACCUM, out), "tv_gemm_small_fwd"),
                                       (lambda: ops.norm_shift(r(4, 96, dtype=F32), r(1), 1e-5, shift=r(96), state=state, plan=p), "tv_norm_shift_fwd"),
                                       (lambda: ops.rms_norm(x, r(512), 1e-5), "tv_rmsnorm_fwd"))):
        with pytest.raises(ops.TimeViperHipError, match=f"^{entry} failed .status -4.: an earlier call's"):
            call()
        assert failing.value == n + 1
    assert torch.equal(out, before) and torch.equal(state, state0)


@pytest.mark.gpu
def test_threads_on_streams_of_their_own():
    x, w = [r(64 + i, 1024, seed=i) for i in range(4)], r(1024)
    want = [ops.rms_norm(v, w, 1e-5) for v in x]
    torch.cuda.synchronize()
    ok = [False] * 4

    def go(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                y = ops.rms_norm(x[i], w, 1e-5)
            torch.cuda.current_stream().synchronize()
            ok[i] = torch.equal(y, want[i])
    threads = [threading.Thread(target=go, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(ok)


@pytest.mark.gpu
def test_the_order_of_a_side_stream():
    """A producer that is still at work on a side stream, the operators, a consumer there, without a wait between: launched anywhere else, an operator would read what was there before"""
    slow, w, m, out = r(4096, 4096) * 2 ** -6, r(512), r(640, 512), []
    want = [ops.rms_norm(r(200, 512, seed=i), w, 1e-5) for i in range(6)]
    want = [(a, ops.mid_linear(a, m), ops.flash_attn_func(*[a.view(1, 50, 4, 512)[..., j * 64:j * 64 + 64] for j in range(3)])) for a in want]
    values = [r(200, 512, seed=i) for i in range(6)]
    x = torch.zeros(200, 512, dtype=BF, device=DEV)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for v in values:
            y = slow
            for _ in range(24):                                                          # (some milliseconds: the host is far ahead)
                y = y @ slow
            x.copy_(v + 0 * y.flatten()[:1].nan_to_num(0, 0, 0))
            a = ops.rms_norm(x, w, 1e-5)
            b = ops.mid_linear(a, m)
            c = ops.flash_attn_func(*[a.view(1, 50, 4, 512)[..., j * 64:j * 64 + 64] for j in range(3)])
            out.append((a.clone(), b.clone(), c.clone()))
            del a, b, c                                                                  # (their memory is the next step's)
            x.zero_()
    side.synchronize()
    for got, exp in zip(out, want):
        assert all(torch.equal(g, e) for g, e in zip(got, exp))


@pytest.mark.parametrize("name", NAMES)
def test_nothing_but_gpu_tensors(name):
    """CPU tensors, no tensors, too few arguments: None, and no error left behind"""
    f = getattr(native, name)
    t = torch.ones(2, 4, 8, 8, dtype=torch.bfloat16)
    assert f() is None and all(f(*[v] * n) is None for v in (t, None, 1, "a") for n in range(1, 18))
