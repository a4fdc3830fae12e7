"""The fp32 scan on the matrix cores (csrc/ssd_f32.hip) against chunks in 64 bits: ends of chunks and of segments, segments of one chunk and of several, operands that
keep the general kernels."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(x, d, A, Bm, Cm, D, S, of):
    """(y, final state, magnitudes of both): x (B, L, H, P) ... in 64 bits, 32 tokens at a time"""
    L, H = x.shape[1:3]
    y, mag, Sm = torch.empty_like(x), torch.empty_like(x), S.abs()
    for t in range(0, L, 32):
        xt, dt, b, c = (v[:, t:t + 32].transpose(1, 2).contiguous() for v in (x, d, Bm[:, :, of], Cm[:, :, of]))
        cs = torch.cumsum(dt * A[:, None], 2)
        M = torch.exp((cs[..., :, None] - cs[..., None, :]).masked_fill(~torch.ones(cs.shape[2], cs.shape[2], dtype=torch.bool, device=DEV).tril(), -float("inf")))
        xd, bt, e, w = xt * dt[..., None], b.transpose(2, 3).contiguous(), torch.exp(cs)[..., None], torch.exp(cs[..., -1:] - cs)[..., None]
        for o, f, s in ((y, lambda v: v, S), (mag, torch.abs, Sm)):
            o[:, t:t + 32] = (torch.matmul(M * torch.matmul(f(c), f(bt)), f(xd)) + e * torch.matmul(f(c), s.transpose(2, 3).contiguous())
                              + f(D)[:, None, None] * f(xt)).transpose(1, 2)
        step = lambda f, s: torch.exp(cs[..., -1])[..., None, None] * s + torch.matmul((f(xd) * w).transpose(2, 3).contiguous(), f(b))
        S, Sm = step(lambda v: v, S), step(torch.abs, Sm)
    return y, S, mag, Sm


@pytest.mark.parametrize("B,L,H,P,G,group_map,init", [(1, 65, 2, 16, 1, "block", True), (2, 128, 4, 48, 2, "tile", False), (1, 129, 4, 64, 4, "block", True),
                                                      (2, 1000, 32, 128, 2, "block", True), (1, 4096, 32, 64, 2, "tile", False)])
@pytest.mark.parametrize("form", ["dense", "rows", "general"])
def test_against_64_bits(B, L, H, P, G, group_map, init, form):
    """rows: operands as slices of wider rows; general: rows off the 16-byte pieces"""
    from timeviper_amd import kernels as ops
    N = 16
    g = torch.Generator(device=DEV).manual_seed(L + P)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    off = {"dense": 0, "rows": 8, "general": 3}[form]
    wide = lambda *s: r(*s[:2], s[2] * s[3] + off)[..., off:].unflatten(2, s[2:])
    x, Bm, Cm = wide(B, L, H, P), 0.3 * r(B, G, L, N + off)[..., off:].transpose(1, 2), wide(B, L, G, N)
    dt, A, bias, D = r(B, L, H), -torch.linspace(0.01, 8, H, device=DEV), torch.linspace(-4, 0, H, device=DEV), r(H)
    S0 = r(B, H, P, N) if init else None
    y, fin, dec = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=S0, return_final_states=True,
                                                return_total_decay=True, group_map=group_map)
    assert ops.ssd_scan_last_kernel() == (8 if form == "general" else 11)
    of = torch.arange(H, device=DEV) % G if group_map == "tile" else torch.arange(H, device=DEV) // (H // G)
    d = F.softplus(dt.double() + bias.double())
    want, S, mag, Sm = reference(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), torch.zeros(B, H, P, N, device=DEV, dtype=torch.float64)
                                 if S0 is None else S0.double(), of)
    # a few hundred rounded terms (2^-18 of their magnitudes) and exponents that are differences of prefix sums of 64 tokens (2^-21 of the sum)
    rel = 2.0 ** -18 + 2.0 ** -21 * 64 * (d * A.double()).abs().mean(1).max().item()
    assert ((y.double() - want).abs() <= mag * rel + 1e-9).all()
    assert ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5, atol=1e-6)
    if form == "dense":
        only = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=S0, group_map=group_map)
        assert torch.equal(only, y)


# the infinity or NaN in the first, an inner and the last token of a 16-token tile; whole and partial chunks, one segment and several
@pytest.mark.parametrize("L,at", [(65, 0), (130, 21), (130, 129), (512, 303), (500, 495)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_tokens_in_front_of_an_infinity(L, at, value):
    """an x that is no number is not seen by the tokens in front of it, nor by the head's other columns"""
    from timeviper_amd import kernels as ops
    B, H, P, G, N, h, p = 1, 4, 32, 2, 16, 2, 19
    g = torch.Generator(device=DEV).manual_seed(L + at)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, Bm, Cm, dt = r(B, L, H, P), 0.3 * r(B, L, G, N), r(B, L, G, N), r(B, L, H)
    A, bias, D = -torch.linspace(0.01, 2, H, device=DEV), torch.linspace(-4, 0, H, device=DEV), r(H)
    f = lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, return_final_states=True)
    clean, S = f()
    x[0, at, h, p] = value
    y, fin = f()
    assert ops.ssd_scan_last_kernel() == 11
    hit = torch.zeros(B, L, H, P, dtype=torch.bool, device=DEV)
    hit[0, at:, h, p] = True
    # (the tile is summed in another order: 16 terms, each within 2^-24 of the magnitudes, which are below 100 here)
    assert (y[~hit] - clean[~hit]).abs().max() < 1e-3 and not torch.isfinite(y[0, at, h, p]) and not torch.isfinite(fin[0, h, p]).any()
    keep = torch.ones(B, H, P, dtype=torch.bool, device=DEV)
    keep[0, h, p] = False
    assert torch.equal(fin[keep], S[keep])


# 7 | 8 chunks (one | two work-groups a tile), a second one with fewer segments than waves, more chunks a segment than stay in LDS, 16 blocks' remainders, a column tile of a round more
@pytest.mark.parametrize("B,L,H,P", [(1, 448, 32, 64), (1, 449, 32, 64), (1, 520, 2, 16), (1, 1039, 32, 64), (1, 2100, 16, 64), (1, 4096, 4, 32), (2, 1010, 16, 64), (2, 1010, 33, 64),
                                     (1, 70, 5, 48), (3, 330, 40, 32), (1, 6000, 8, 32)])
@pytest.mark.parametrize("group_map", ["block", "tile"])
def test_work_groups_of_a_tile(B, L, H, P, group_map):
    from timeviper_amd import kernels as ops
    G = 1 if H % 2 else 2
    g = torch.Generator(device=DEV).manual_seed(L + H)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, Bm, Cm, dt, D, S0 = r(B, L, H, P), 0.3 * r(B, L, G, 16), r(B, L, G, 16), r(B, L, H), r(H), r(B, H, P, 16)
    A = -torch.linspace(1e-3, 4, H, device=DEV)
    y, fin, dec = ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_softplus=True, initial_states=S0, return_final_states=True, return_total_decay=True, group_map=group_map)
    assert ops.ssd_scan_last_kernel() == 11
    d = F.softplus(dt.double())
    of = torch.arange(H, device=DEV) % G if group_map == "tile" else torch.arange(H, device=DEV) // (H // G)
    want, S, mag, Sm = reference(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), S0.double(), of)
    # (as above; exponents are sums of 16 tokens)
    rel = 2.0 ** -18 + 2.0 ** -21 * 16 * (d * A.double()).abs().mean(1).max().item()
    assert ((y.double() - want).abs() <= mag * rel + 1e-9).all() and ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5, atol=1e-6)


# two launches (csrc/ssd_f32_long.hip): each side of its lines in tiles (batch x heads x head_dim / 16) and chunks, partial chunks and a last segment of one, infinities
@pytest.mark.parametrize("B,L,H,P,two", [(1, 1472, 8, 64, False), (1, 1473, 8, 64, True), (2, 3777, 8, 64, True), (2, 3776, 8, 64, False), (1, 4097, 20, 64, True), (1, 4097, 21, 64, False),
                                         (1, 4128, 65, 64, True), (1, 4128, 85, 64, False), (1, 7700, 33, 64, True), (3, 2000, 1, 48, True), (1, 5000, 1, 16, True), (2, 1900, 512, 64, True)])
def test_two_launches(B, L, H, P, two):
    from timeviper_amd import _capi
    from timeviper_amd import kernels as ops
    G, n = 1 if H % 2 else 2, _capi.lib().tv_ssd_scan_workspace_bytes
    # (beyond 4 096 tokens nothing else asks for more than a place to point to)
    assert L <= 4096 or (n(B, L, H, P, G, 16, ops.TV_F32) > 256) == two
    g = torch.Generator(device=DEV).manual_seed(L + H)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, Bm, Cm, dt, D, S0 = r(B, L, H, P), 0.3 * r(B, L, G, 16), r(B, L, G, 16), r(B, L, H), r(H), r(B, H, P, 16)
    A = -torch.linspace(1e-3, 4, H, device=DEV)
    call = lambda: ops.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_softplus=True, initial_states=S0, return_final_states=True, return_total_decay=True)
    y, fin, dec = call()
    assert ops.ssd_scan_last_kernel() == 11
    d = F.softplus(dt.double())
    if B * L * H * P < 1e7:
        want, S, mag, Sm = reference(x.double(), d, A.double(), Bm.double(), Cm.double(), D.double(), S0.double(), torch.arange(H, device=DEV) // (H // G))
        # (as above: exponents are differences of sums of at most 64 tokens)
        rel = 2.0 ** -18 + 2.0 ** -21 * 64 * (d * A.double()).abs().mean(1).max().item()
        assert ((y.double() - want).abs() <= mag * rel + 1e-9).all() and ((fin.double() - S).abs() <= Sm * rel + 1e-9).all()
    else:
        # heads do not depend on each other: the last four of them alone, on the other kernel
        part = ops.mamba_chunk_scan_combined(x[:, :, -4:].contiguous(), dt[:, :, -4:].contiguous(), A[-4:], Bm[:, :, -1:].contiguous(), Cm[:, :, -1:].contiguous(), D=D[-4:], dt_softplus=True,
                                             initial_states=S0[:, -4:].contiguous(), return_final_states=True)
        assert (y[:, :, -4:] - part[0]).norm() <= 2e-6 * part[0].norm() and (fin[:, -4:] - part[1]).norm() <= 2e-6 * part[1].norm()
    assert torch.allclose(dec.double(), (d * A.double()).sum(1), rtol=1e-5, atol=1e-6)
    at = L // 2
    x[0, at, H - 1, 3] = float("inf")
    z, _, _ = call()
    assert torch.isfinite(z[:, :at]).all() and torch.isfinite(z[..., :3]).all() and not torch.isfinite(z[0, at, H - 1, 3])
