"""The chunk-parallel scan of small states (csrc/ssd_chunked.hip) against the token recurrence in 64 bits, at the edges of its tiles."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


# last chunk of one and of 63 tokens; columns and states that are no multiple of 4, more than 64 columns, 64 states; every dtype it takes
@pytest.mark.parametrize("L", [65, 127, 128, 500])
@pytest.mark.parametrize("P,N", [(64, 16), (30, 5), (100, 33), (128, 64), (1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_chunked(L, P, N, dtype):
    from timeviper_amd import kernels as ops
    B, H, G = 2, 4, 2
    g = torch.Generator(device=DEV).manual_seed(L + P + N)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, Bm, Cm = r(B, L, H, P).to(dtype), (0.3 * r(B, L, G, N)).to(dtype), (0.3 * r(B, L, G, N)).to(dtype)
    dt, A, bias, D = r(B, L, H).to(dtype), -torch.linspace(0.01, 8, H, device=DEV), torch.linspace(-4, 0, H, device=DEV), r(H)
    init = r(B, H, P, N)
    ops.ssd_scan_set_impl(8)                                   # (some of these have a form on the matrix cores, csrc/ssd_f32.hip)
    try:
        y, fin, dec = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=True,
                                                    return_total_decay=True)
    finally:
        ops.ssd_scan_set_impl(0)
    assert ops.ssd_scan_last_kernel() == 8
    of = torch.arange(H, device=DEV) // (H // G)
    d = F.softplus(dt.double() + bias.double())
    S, want, mag = init.double(), torch.empty(B, L, H, P, device=DEV, dtype=torch.float64), torch.empty(B, L, H, P, device=DEV, dtype=torch.float64)
    Sm = S.abs()
    for t in range(L):
        e, b, c, xt = torch.exp(d[:, t] * A.double())[..., None, None], Bm[:, t, of].double(), Cm[:, t, of].double(), x[:, t].double()
        S = e * S + (d[:, t, :, None] * xt)[..., None] * b[:, :, None]
        Sm = e * Sm + ((d[:, t, :, None] * xt)[..., None] * b[:, :, None]).abs()
        want[:, t] = (S * c[:, :, None]).sum(-1) + D[:, None] * xt
        mag[:, t] = (Sm * c[:, :, None].abs()).sum(-1) + (D[:, None] * xt).abs()
    # fp32: a few hundred rounded terms (2^-18 of their magnitudes) and exponents that are differences of prefix sums of 64 tokens (each
    # off by some 2^-24 of the sum a step: 2^-21 of it); a bf16 y is rounded twice
    rel = 2.0 ** -18 + 2.0 ** -21 * 64 * (d * A.double()).abs().mean(1).max().item()
    tol = mag * rel + (0 if dtype is torch.float32 else 2.0 ** -8 * (2 * want.abs() + mag))
    assert ((y.double() - want).abs() <= tol + 1e-9).all()
    assert ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5, atol=1e-6)
