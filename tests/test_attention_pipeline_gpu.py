"""Attention's software pipeline: maxima and accumulators that follow tile by tile, the ring's halves, runs of tiles that a window leaves out; one and two waves a query row."""
import math

import pytest
import torch

from test_attention_two_waves_gpu import close, reference

pytestmark = pytest.mark.gpu
DEV = "cuda"


# tiles of 64 keys, two a step, four places a ring: a length for every remainder; B x H pairs: two waves a row, and (more than a round of blocks of either size) one
@pytest.mark.parametrize("pairs", [(1, 2), (90, 4)])
@pytest.mark.parametrize("D,Lq,Lk,causal,dtype", [(128, 257, 257, True, torch.bfloat16), (128, 320, 511, True, torch.bfloat16), (128, 300, 64, False, torch.bfloat16), (128, 270, 128, False, torch.bfloat16),
                                                  (64, 300, 129, False, torch.bfloat16), (96, 257, 192, False, torch.bfloat16), (80, 258, 577, True, torch.bfloat16), (72, 300, 321, True, torch.float16),
                                                  (128, 300, 200, True, torch.float16), (128, 513, 513, True, torch.bfloat16)])
def test_rising_scores(D, Lq, Lk, causal, dtype, pairs):
    """Scores that rise and fall along the keys by hundreds of powers of two: the accumulators are rescaled at some tiles and not at others"""
    from timeviper_amd import kernels as ops
    B, H = pairs
    g = torch.Generator(device=DEV).manual_seed(Lq * 1000 + Lk + D)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    u = torch.nn.functional.normalize(r(D), dim=0) * D ** 0.5
    rise = torch.linspace(-4, 4, Lk, device=DEV) + 3 * torch.sin(torch.arange(Lk, device=DEV) / 37.0)
    slope = torch.linspace(-6, 6, Lq, device=DEV)                       # falling rows, level rows, rising rows
    q = (r(B, Lq, H, D) + slope[None, :, None, None] * u).to(dtype)
    k = (r(B, Lk, H, D) + rise[None, :, None, None] * u).to(dtype)
    v = r(B, Lk, H, D).to(dtype)
    pos, key = torch.arange(Lq, device=DEV)[:, None] + (Lk - Lq), torch.arange(Lk, device=DEV)[None]
    ok = key <= pos if causal else torch.ones(Lq, Lk, dtype=torch.bool, device=DEV)
    got, lse = ops.flash_attn_func(q, k, v, causal=causal, return_lse=True)
    want, wlse, mag = reference(q, k, v, ok, D ** -0.5)
    # a score is a sum of D products in fp32: off by D 2^-24 |q| |k| scale at most (the products cancel; scores reach 200), and so is lse, to which m ln 2 + log(l) adds three
    # roundings; a weight is off by twice that as a factor, beside its rounding and the result's (`close`)
    e = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    off = D * 2.0 ** -24 * float(q.double().norm(dim=3).max() * k.double().norm(dim=3).max()) * D ** -0.5
    assert off < 5e-3 and ((got.double() - want).abs() <= (1.05 * e + 2.1 * off) * (mag + want.abs()) + 2e-3 * e).all()
    some = torch.isfinite(wlse)
    assert torch.equal(torch.isfinite(lse), some) and ((lse.double() - wlse)[some].abs() <= off + 2.0 ** -22 * (1 + wlse[some].abs())).all()


# kept keys, then a gap of an even and of an odd number of tiles, none at all, and one that is inside a step of two tiles; few heads (two waves a row) and many
@pytest.mark.parametrize("H", [2, 64])
@pytest.mark.parametrize("D,counts,starts,window,keep", [(128, [300, 270], [0, 900], 192, 64), (128, [300, 270], [0, 837], 190, 65), (128, [700], [0], 256, 1), (64, [513], [1000], 128, 200),
                                                         (96, [260, 5], [330, 700], 320, 64), (128, [300], [200], 333, 130)])
def test_gaps(D, counts, starts, window, keep, H):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm.cache import SlotStateCache
    G, n = 2, len(counts)
    g = torch.Generator(device=DEV).manual_seed(sum(counts) + window)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    cache = SlotStateCache([("tokens", 2 * G * D)], n, torch.bfloat16, DEV, max(a + c for a, c in zip(starts, counts)))
    slots = [cache.alloc() for _ in counts]
    if any(starts):
        cache.commit(cache.plan([s for s, a in zip(slots, starts) if a], [a for a in starts if a]))
    plan, rows = cache.plan(slots, counts), cache.tokens(0)
    rows.copy_(r(*rows.shape))
    q = r(sum(counts), H, D)
    got = ops.attention_window(q, rows, plan, G, D ** -0.5, window=window, keep_first=keep)
    at = 0
    for s, c, a in zip(slots, counts, starts):
        kv = rows[s, :a + c].view(1, a + c, 2, G, D)
        pos, key = torch.arange(a, a + c, device=DEV)[:, None], torch.arange(a + c, device=DEV)[None]
        want, _, mag = reference(q[None, at:at + c], kv[:, :, 0], kv[:, :, 1], (key <= pos) & ((key > pos - window) | (key < keep)), D ** -0.5)
        close(got[None, at:at + c], want, mag)
        at += c
