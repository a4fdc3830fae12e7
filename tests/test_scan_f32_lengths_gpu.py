"""The fp32 scan on the matrix cores at the lengths around those of the chunked kernels: 48 to 64 tokens and more than 4 096; decays that are fast, slow, and that reset a head."""
import pytest
import torch
import torch.nn.functional as F

from test_scan_f32_gpu import reference

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(B, L, H, P, G, decays, off=0):
    g = torch.Generator(device=DEV).manual_seed(L + P)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    wide = lambda *s: r(*s[:2], s[2] * s[3] + off)[..., off:].unflatten(2, s[2:])
    x, Bm, Cm, dt = wide(B, L, H, P), 0.3 * wide(B, L, G, 16), wide(B, L, G, 16), r(B, L, H)
    A, bias, D = -torch.linspace(0.5, 8, H, device=DEV), torch.zeros(H, device=DEV), r(H)
    if decays == "slow":
        A = A * 1e-3
    elif decays == "reset":                       # one token in eight leaves nothing of what was before it
        dt = torch.where(torch.rand(B, L, H, generator=g, device=DEV) < .125, dt.abs() * 1e4, dt - 6)
    return x, dt, A, Bm, Cm, D, bias, r(B, H, P, 16)


@pytest.mark.parametrize("B,L,H,P,G", [(1, 1, 8, 64, 2), (2, 15, 8, 64, 2), (2, 47, 8, 64, 2), (1, 48, 6, 16, 3), (3, 49, 4, 80, 1), (1, 63, 8, 128, 8), (2, 64, 8, 64, 2), (1, 64, 4, 256, 1),
                                       (1, 4097, 4, 32, 2), (1, 4160, 4, 32, 2), (2, 9000, 2, 16, 1)])
@pytest.mark.parametrize("decays", ["fast", "slow", "reset"])
@pytest.mark.parametrize("init", [False, True])
def test_against_64_bits(B, L, H, P, G, decays, init):
    from timeviper_amd import kernels as ops
    x, dt, A, Bm, Cm, D, bias, S0 = operands(B, L, H, P, G, decays, 8 if L % 2 else 0)
    y, fin, dec = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=S0 if init else None, return_final_states=True,
                                                return_total_decay=True)
    assert ops.ssd_scan_last_kernel() == (11 if L >= 48 else 1)
    d = F.softplus(dt.double())
    want, S, mag, Sm = reference(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), S0.double() if init else torch.zeros_like(S0).double(), torch.arange(H, device=DEV) // (H // G))
    # a few hundred rounded terms (2^-18 of their magnitudes); an exponent of a token's dt A and of sums that keep what they lose is off by some 2^-22 of itself: of a weight
    # e^-s that is s e^-s 2^-22, below the terms' own; the state's weights are sums from the end
    rel = 2.0 ** -18
    assert ((y.double() - want).abs() <= mag * rel + 1e-9).all()
    assert ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("L,at", [(48, 0), (50, 17), (64, 63), (4100, 70)])
@pytest.mark.parametrize("what", ["x", "B", "C", "dt"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_before_what_is_no_number(L, at, what, value):
    """tokens in front of it and other heads' (groups') rows are as without it; its own token is none either, but for a dt, which is clamped first (a NaN to its lower end)"""
    from timeviper_amd import kernels as ops
    x, dt, A, Bm, Cm, D, bias, S0 = operands(1, L, 4, 32, 2, "slow")
    f = lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=S0)
    clean = f()
    {"x": x[0, at, 2], "B": Bm[0, at, 1], "C": Cm[0, at, 1], "dt": dt[0, at, 2:3]}[what][:] = value
    y = f()
    assert ops.ssd_scan_last_kernel() == 11
    heads = [0, 1] if what in ("B", "C") else [0, 1, 3]
    # (where x is no number its tile of 16 tokens is summed in another order)
    near = lambda a, b: (a - b).abs().max() < 1e-3 if a.numel() else True
    assert near(y[:, :, heads], clean[:, :, heads]) and near(y[:, :at], clean[:, :at]) and (what == "dt" or not torch.isfinite(y[0, at, 2]).any())
    if what == "C":
        assert near(y[:, at + 1:], clean[:, at + 1:])
    if what == "dt" and value != value:
        ops.ssd_scan_set_impl(1)
        try:
            z = f()
            assert ops.ssd_scan_last_kernel() == 1
        finally:
            ops.ssd_scan_set_impl(0)
        d = F.softplus(dt.double()).nan_to_num(0.0)
        mag = reference(x.double(), d, *(v.double() for v in (A, Bm, Cm, D, S0)), torch.arange(4, device=DEV) // 2)[2]
        assert ((y - z).abs() <= 2 * 2.0 ** -18 * mag).all()               # (both within 2^-18 of the terms, as above)


@pytest.mark.parametrize("B,L,H,P", [(2, 3000, 32, 64), (1, 2100, 32, 64), (2, 700, 128, 64), (2, 1300, 24, 64)])
def test_segments_of_a_round(B, L, H, P):
    """segments that are as many as fill a round, and that begin another one"""
    from timeviper_amd import kernels as ops
    x, dt, A, Bm, Cm, D, bias, S0 = operands(B, L, H, P, 2, "slow")
    y, fin = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=S0, return_final_states=True)
    assert ops.ssd_scan_last_kernel() == 11
    d = F.softplus(dt.double())
    want, S, mag, Sm = reference(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), S0.double(), torch.arange(H, device=DEV) // (H // 2))
    # (as test_scan_f32_gpu.py: exponents are differences of prefix sums of 64 tokens, here below 1)
    rel = 2.0 ** -18 + 2.0 ** -21 * 64 * (d * A.double()).abs().mean(1).max().item()
    assert ((y.double() - want).abs() <= mag * rel + 1e-9).all() and ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()


def stepwise(x, d, A, Bm, Cm, D, S, of):
    """`reference` token by token: no sums of exponents, of which an endless step leaves nothing"""
    y, mag, Sm = torch.empty_like(x), torch.empty_like(x), S.abs()
    for t in range(x.shape[1]):
        e, xd, b, c = torch.exp(d[:, t] * A)[..., None, None], (d[:, t, :, None] * x[:, t])[..., None], Bm[:, t, of][:, :, None], Cm[:, t, of][:, :, None]
        S, Sm = e * S + xd * b, e * Sm + (xd * b).abs()
        y[:, t], mag[:, t] = (S * c).sum(-1) + D[:, None] * x[:, t], (Sm * c.abs()).sum(-1) + (D[:, None] * x[:, t]).abs()
    return y, S, mag, Sm


@pytest.mark.parametrize("L,at", [(48, (0,)), (50, (17, 18)), (64, (5, 31, 63)), (4100, (70,)), (4160, (0, 64, 4098, 4100))])
@pytest.mark.parametrize("init", [False, True])
@pytest.mark.parametrize("step", [float("inf"), 3e38, 1e7])
def test_a_step_that_resets_without_end(L, at, init, step):
    """an infinite dt (or one whose product with B is no number) where x is 0 empties the state, and what follows is as after any token: nothing but numbers"""
    from timeviper_amd import kernels as ops
    H = 4
    x, dt, A, Bm, Cm, D, bias, S0 = operands(1, L, H, 32, 2, "fast")
    dt = dt.abs() * .1
    dt[0, list(at)], x[0, list(at)] = step, 0.
    y, fin, dec = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, initial_states=S0 if init else None, return_final_states=True, return_total_decay=True)
    assert ops.ssd_scan_last_kernel() == 11
    d = dt.double().clamp(max=3.0e38)
    want, S, mag, Sm = stepwise(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), S0.double() if init else torch.zeros_like(S0).double(), torch.arange(H, device=DEV) // 2)
    rel = 2.0 ** -18                                                       # (as above)
    assert ((y.double() - want).abs() <= mag * rel + 1e-9).all() and ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5) if step < 1e38 else (dec < -1e37).all()


@pytest.mark.parametrize("L,seeds", [(48, 4), (64, 4), (5000, 1)])
@pytest.mark.parametrize("A", [1.0, 0.3, 1e-3, None])
def test_error_is_no_larger_than_token_by_token(L, seeds, A):
    """against 64 bits, in the mean over the elements: y and the state as the recurrence leaves them, or nearer"""
    from timeviper_amd import kernels as ops
    H, errors = 32, {}
    for seed in range(seeds):
        g = torch.Generator(device=DEV).manual_seed(seed)
        r = lambda *s: torch.randn(s, generator=g, device=DEV)
        x, Bm, Cm, dt = r(1, L, H, 64), 0.3 * r(1, L, 2, 16), r(1, L, 2, 16), r(1, L, H)
        Ah, D, S0 = -(torch.linspace(.5, 8, H, device=DEV) if A is None else torch.full((H,), A, device=DEV)), r(H), r(1, H, 64, 16)
        want, S, _, _ = reference(x.double(), F.softplus(dt.double()), Ah.double(), Bm.double(), Cm.double(), D.double(), S0.double(), torch.arange(H, device=DEV) // 16)
        for impl, kernel in ((0, 11), (1, 1)):
            ops.ssd_scan_set_impl(impl)
            try:
                y, fin = ops.mamba_chunk_scan_combined(x, dt, Ah, Bm, Cm, D=D, dt_softplus=True, initial_states=S0, return_final_states=True)
                assert ops.ssd_scan_last_kernel() == kernel
            finally:
                ops.ssd_scan_set_impl(0)
            for what, a, b in (("y", y, want), ("state", fin, S)):
                errors.setdefault((what, kernel), []).append(((a.double() - b).norm() / b.norm()).item())
    for what in ("y", "state"):
        here, there = (sum(errors[what, k]) / seeds for k in (11, 1))
        print(f"{what} {here:.3e} {there:.3e}")
        assert here <= there
