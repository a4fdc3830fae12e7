"""Products of 2..32 rows on the matrix cores (csrc/gemm_skinny.hip) and what a decode step of 5..32 sequences builds on them."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from timeviper_amd import kernels
    return kernels


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV) * scale).bfloat16()


def close(got, x, w, bias=0.0):
    """fp32 sums of bf16 products and one rounding: 2^-8 relative to the value, K 2^-24 relative to the terms"""
    want = x.double() @ w.double().T + bias
    bound = want.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().T) * (x.shape[1] * 2.0 ** -24) + 1e-30
    assert ((got.double() - want).abs() <= bound).all()
    return want


# edges of the 8-row copies, 16-row tiles and 64-column stages; fewer stages than waves; shares of 1, 2, 9, 18 and 32 rows
@pytest.mark.parametrize("M", [2, 5, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N,Kd", [(1, 64), (37, 192), (300, 1024), (4480, 704), (8201, 128), (700, 4480)])
def test_rows_linear(K, M, N, Kd):
    buf = rnd((M, Kd + 24), M + N, 1.0)
    x, w = buf[:, 8:8 + Kd], rnd((N, Kd + 8), 3, Kd ** -0.5)[:, :Kd]
    b = rnd((N,), 4)
    assert K.rows_take(x, w)
    close(K.rows_linear(x, w), x, w)
    y = K.rows_linear(x, w, b)
    close(y, x, w, b.double())
    f = K.rows_linear(x, w, b, out_dtype=torch.float32)
    assert f.dtype == torch.float32 and torch.equal(f.bfloat16(), y)
    assert torch.equal(K.rows_linear(x, w, b, relu2=True), torch.square(torch.relu(y.float())).bfloat16())
    r = torch.randn((M, N), device=DEV)
    xs, h = K.rows_add(x, w, r, b)
    close(xs - r, x, w, b.double()) if N < 64 else None
    assert torch.allclose(xs, r + f, rtol=1e-5, atol=1e-5) and torch.equal(h, xs.bfloat16())


@pytest.mark.parametrize("M", [2, 4, 7, 16, 25])
@pytest.mark.parametrize("n1,ff,Kd", [(3, 1, 64), (130, 77, 192), (1100, 900, 256), (3072, 2500, 512), (40, 0, 128)])
def test_rows_pair(K, M, n1, ff, Kd):
    x, x2, w, b = rnd((M, Kd), 1), rnd((M, Kd), 2), rnd((n1 + 2 * ff, Kd), 3, Kd ** -0.5), rnd((2 * ff,), 4)
    u = torch.full((M, ff + 16), 7.0, device=DEV).bfloat16()
    y = K.rows_pair(x, x2, w, n1, b if ff else None, act_out=u[:, 8:8 + ff])
    close(y, x, w[:n1])
    z = x2.double() @ w[n1:].double().T + b.double()
    want = torch.nn.functional.gelu(z[:, :ff], approximate="tanh") * z[:, ff:]
    assert (u[:, 8:8 + ff].double() - want).abs().max() <= 2.0 ** -8 * want.abs().max() + 1e-4 if ff else True
    assert (u[:, :8] == 7).all() and (u[:, 8 + ff:] == 7).all()


@pytest.mark.parametrize("M", [5, 12, 32])
def test_conv_epilogue_is_the_two_launches(K, M):
    Kd, d_in, C, H = 512, 320, 448, 24
    W, cw, cb = rnd((d_in + C + H, Kd), 1, Kd ** -0.5), rnd((C, 4), 2, 0.5), rnd((C,), 3)
    st_a = rnd((M, C, 4), 4)
    st_b = st_a.clone()
    for step in range(3):
        x = rnd((M, Kd), 10 + step)
        two = K.rows_linear(x, W)
        conv = K.causal_conv1d_update(two[:, d_in:d_in + C], st_a, cw, cb, "silu")
        one = K.rows_linear(x, W, conv=(st_b, cw, cb, d_in))
        assert torch.equal(one[:, d_in:d_in + C], conv) and torch.equal(st_a, st_b)
        assert torch.equal(one[:, :d_in], two[:, :d_in]) and torch.equal(one[:, d_in + C:], two[:, d_in + C:])


def test_refusals(K):
    w = rnd((100, 128), 1)
    assert not K.rows_take(rnd((1, 128), 2), w) and not K.rows_take(rnd((33, 128), 2), w) and not K.rows_take(rnd((4, 128), 2).float(), w)
    assert not K.rows_take(rnd((4, 96), 2), rnd((100, 96), 1)) and not K.rows_take(rnd((4, 128), 2), w.float())
    for bad in (lambda: K.rows_linear(rnd((33, 128), 2), w), lambda: K.rows_linear(rnd((4, 64), 2), w),
                lambda: K.rows_linear(rnd((4, 128), 2), w, bias=torch.zeros(100, device=DEV)),
                lambda: K.rows_linear(rnd((4, 128), 2), w, conv=(rnd((3, 10, 4), 1), rnd((10, 4), 1), None, 0))):
        with pytest.raises(K.TimeViperHipError):
            bad()
    x = rnd((4, 136), 5)[:, 3:131]                       # rows that are not 16-byte aligned are taken by a copy
    close(K.rows_linear(x, w), x, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("P,N", [(80, 128), (24, 24)])
def test_state_update_reads_slices_in_place(K, dtype, P, N):
    B, H, G = 5, 6, 2
    g = torch.Generator(device=DEV).manual_seed(1)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    proj = r(B, 2 * H * P + 2 * G * N + H + 2).to(dtype)
    x, Bm, Cm, dt = proj.split([H * P, G * N, G * N, H, proj.shape[1] - H * P - 2 * G * N - H], 1)[:4]
    st = r(B, H, P, N)
    st2 = st.clone()
    A, D, bias = -torch.rand(H, generator=g, device=DEV) - 0.1, r(H), r(H)
    args = (x.unflatten(1, (H, P)), dt, A, Bm.unflatten(1, (G, N)), Cm.unflatten(1, (G, N)))
    y = K.selective_state_update(st, *args, D, dt_bias=bias, dt_softplus=True)
    y2 = K.selective_state_update(st2, *(t.contiguous() for t in args), D, dt_bias=bias, dt_softplus=True)
    assert torch.equal(y, y2) and torch.equal(st, st2)


@pytest.mark.parametrize("B,far", [(1, (0, 1, 2, 3)), (3, (0,)), (3, (1,)), (3, (2,)), (3, (3,))])
def test_state_update_of_one_sequence_and_of_single_operands_apart(K, B, far):
    """x, dt, B, C (by number) with sequences further apart than dense, the others dense; one sequence has no distance"""
    H, G, P, N = 6, 2, 80, 128
    g = torch.Generator(device=DEV).manual_seed(2)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    widths = (H * P, H, G * N, G * N)
    flat = [r(B, n + 8 * (i in far)).bfloat16()[:, :n] for i, n in enumerate(widths)]
    A, D, bias, st = -torch.rand(H, generator=g, device=DEV) - 0.1, r(H), r(H), r(B, H, P, N)
    st2 = st.clone()
    step = lambda s, t: K.selective_state_update(s, t[0].unflatten(1, (H, P)), t[1], A, t[2].unflatten(1, (G, N)), t[3].unflatten(1, (G, N)), D,
                                                 dt_bias=bias, dt_softplus=True)
    assert torch.equal(step(st, flat), step(st2, [t.contiguous() for t in flat])) and torch.equal(st, st2)


def test_state_update_refuses_an_empty_batch(K):
    z = lambda *s: torch.zeros(s, device=DEV)
    with pytest.raises(K.TimeViperHipError):
        K.selective_state_update(z(0, 2, 16, 16), z(0, 2, 16), z(0, 2), z(2), z(0, 1, 16), z(0, 1, 16))


@pytest.mark.parametrize("B", [5, 17])
def test_decode_step_of_many_sequences_is_the_general_one(K, B, monkeypatch):
    """5..32 sequences on tv_gemm_rows_fwd against torch.nn.Linear and the stand-alone operators: same rounding points"""
    from timeviper_amd.model.llm.nano import HybridMambaAttentionDynamicCache, NemotronHConfig, NemotronHForCausalLM
    cfg = NemotronHConfig(vocab_size=256, hidden_size=256, intermediate_size=384, num_hidden_layers=6, hybrid_override_pattern="M-*M-*",
                          num_attention_heads=4, head_dim=128, num_key_value_heads=2, ssm_state_size=16, mamba_num_heads=8,
                          mamba_n_groups=2, mamba_head_dim=16, mamba_chunk_size=16)
    torch.manual_seed(0)
    model = NemotronHForCausalLM(cfg).bfloat16().to(DEV).eval()
    g = torch.Generator(device=DEV).manual_seed(9)
    prompt = torch.randint(0, 256, (B, 40), device=DEV, generator=g)
    forced = torch.randint(0, 256, (4, B, 1), device=DEV, generator=g)
    one, runs = torch.ones(1, dtype=torch.long), {}
    for mode in ("0", "1"):
        monkeypatch.setenv("TV_DECODE_FUSED", mode)
        calls = []
        orig = K.rows_linear
        monkeypatch.setattr(K, "rows_linear", lambda *a, **kw: (calls.append(1), orig(*a, **kw))[1])
        with torch.inference_mode():
            cache = HybridMambaAttentionDynamicCache(cfg, B, dtype=torch.bfloat16, device=DEV)
            model(input_ids=prompt, past_key_values=cache, use_cache=True, cache_position=torch.zeros(1, dtype=torch.long))
            del calls[:]
            outs = [model(input_ids=t, past_key_values=cache, use_cache=True, cache_position=one).logits[:, -1].clone() for t in forced]
        monkeypatch.setattr(K, "rows_linear", orig)
        runs[mode] = (outs, cache, len(calls))
    assert runs["0"][2] == 0 and runs["1"][2] == 4 * (2 * 3 * 2 + 1)
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    assert all(rel(a, b) < 2e-2 for a, b in zip(runs["1"][0], runs["0"][0]))
    c0, c1 = runs["0"][1], runs["1"][1]
    for i in range(6):
        if c0.ssm_states[i].numel():
            assert rel(c1.ssm_states[i], c0.ssm_states[i]) < 2e-2 and rel(c1.conv_states[i], c0.conv_states[i]) < 2e-2
