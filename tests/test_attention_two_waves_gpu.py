"""Attention with two waves a query row (128-row blocks, every second key tile a wave): edges of blocks, of tiles and of steps of two tiles."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, k, v, ok, scale, sink=None):
    """(result, log-sum-exp, sum of |weight x value|) in 64 bits; ok (Lq, Lk): visible keys"""
    B, Lq, H, D = q.shape
    rep = H // k.shape[2]
    q, k, v = (t.double().transpose(1, 2).contiguous() for t in (q, k.repeat_interleave(rep, 2), v.repeat_interleave(rep, 2)))
    s = (torch.matmul(q, k.transpose(2, 3).contiguous()) * scale).masked_fill(~ok, -math.inf)
    lse = torch.logsumexp(s if sink is None else torch.cat([s, sink.double().view(1, H, 1, 1).expand(B, H, Lq, 1)], 3), 3)
    p = torch.exp(s - lse[..., None]).nan_to_num(0.0)
    return torch.matmul(p, v).transpose(1, 2), lse, torch.matmul(p, v.abs()).transpose(1, 2)


def close(got, want, mag):
    # weights and result rounded (2^-8 each for bf16, 2^-11 for f16); scores of fp32 sums
    e = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -11
    assert ((got.double() - want).abs() <= 1.05 * e * (mag + want.abs()) + 2e-3 * e).all(), (got.double() - want).abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,G,D,Lq,Lk,causal", [
    (1, 4, 2, 128, 1, 1, True), (1, 4, 2, 128, 2, 63, True), (2, 4, 4, 128, 31, 64, True), (1, 8, 2, 128, 33, 65, True), (1, 4, 1, 128, 127, 128, True),
    (1, 4, 1, 128, 128, 129, False), (1, 2, 2, 128, 129, 129, True), (1, 2, 1, 128, 257, 191, True), (1, 2, 1, 128, 100, 20, True), (1, 3, 3, 72, 255, 193, False),
    (2, 3, 3, 64, 300, 300, True), (1, 2, 2, 96, 140, 1000, True), (1, 2, 2, 80, 64, 513, False), (70, 1, 1, 64, 100, 100, False), (1, 16, 4, 128, 1000, 1000, True),
    # more than a round of 128-row blocks: where the longest ones' time is filled up, and where not
    (1, 44, 11, 64, 1100, 1100, True), (50, 4, 1, 128, 129, 130, True), (32, 4, 2, 80, 257, 257, True), (20, 5, 1, 64, 400, 490, True),
    # short sequences: one wave a row where the keys are one tile of 96, up to a round of them and beyond
    (1, 2, 1, 64, 96, 96, False), (1, 2, 1, 72, 1, 96, True), (2, 4, 2, 80, 128, 96, True), (1, 4, 1, 128, 100, 66, True), (1, 2, 2, 64, 64, 64, False), (3, 2, 1, 96, 3, 90, False),
    (300, 2, 2, 128, 96, 96, False), (150, 4, 1, 128, 70, 65, False), (150, 4, 1, 128, 70, 64, False), (600, 1, 1, 80, 1, 1, True), (300, 2, 1, 64, 65, 65, True), (200, 3, 3, 72, 96, 96, False), (130, 4, 2, 96, 128, 96, True), (513, 1, 1, 64, 33, 20, True),
    (513, 1, 1, 64, 100, 97, True)])
def test_against_64_bits(B, H, G, D, Lq, Lk, causal, dtype):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(Lq * 1000 + Lk)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)
    q, k, v = r(B, Lq, H, D), r(B, Lk, G, D), r(B, Lk, G, D)
    pos, key = torch.arange(Lq, device=DEV)[:, None] + (Lk - Lq), torch.arange(Lk, device=DEV)[None]
    ok = key <= pos if causal else torch.ones(Lq, Lk, dtype=torch.bool, device=DEV)
    got, lse = ops.flash_attn_func(q, k, v, causal=causal, return_lse=True)
    want, wlse, mag = reference(q, k, v, ok, D ** -0.5)
    close(got, want, mag)
    some = torch.isfinite(wlse)
    assert torch.equal(torch.isfinite(lse), some) and ((lse.double() - wlse)[some].abs() <= 1e-4 * (1 + wlse[some].abs())).all()


# windows that end inside a tile, kept keys, sequences in one launch; chunks behind a cache
@pytest.mark.parametrize("counts,starts,window,keep", [([1, 64, 127], [0, 0, 0], 50, 0), ([128, 33], [70, 500], 100, 7), ([300], [0], 128, 64), ([257, 1], [0, 640], 191, 65),
                                                       ([130], [400], 2 ** 31 - 1, 0), ([1400] * 6, [0] * 6, 1024, 64), ([520] * 14, [0] * 14, 200, 1)])
def test_windows(counts, starts, window, keep):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm.cache import SlotStateCache
    H, G, D, n = 4, 2, 128, len(counts)
    g = torch.Generator(device=DEV).manual_seed(sum(counts))
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    cache = SlotStateCache([("tokens", 2 * G * D)], n, torch.bfloat16, DEV, max(a + c for a, c in zip(starts, counts)))
    slots = [cache.alloc() for _ in counts]
    if any(starts):
        cache.commit(cache.plan([s for s, a in zip(slots, starts) if a], [a for a in starts if a]))
    plan, rows = cache.plan(slots, counts), cache.tokens(0)
    rows.copy_(r(*rows.shape))
    T = sum(counts)
    q, gate = r(T, H, D), r(T, H, D)
    got = ops.attention_window(q, rows, plan, G, D ** -0.5, window=window, keep_first=keep, gate=gate)
    at = 0
    for s, c, a in zip(slots, counts, starts):
        kv = rows[s, :a + c].view(1, a + c, 2, G, D)
        pos, key = torch.arange(a, a + c, device=DEV)[:, None], torch.arange(a + c, device=DEV)[None]
        want, _, mag = reference(q[None, at:at + c], kv[:, :, 0], kv[:, :, 1], (key <= pos) & ((key > pos - window) | (key < keep)), D ** -0.5)
        f = torch.sigmoid(gate[None, at:at + c].double())
        close(got[None, at:at + c], want * f, mag * f)
        at += c


def test_sink():
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(7)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    q, k, v, sink = r(200, 4, 128), r(1, 330, 2, 128), r(1, 330, 2, 64), torch.randn(4, generator=g, device=DEV)
    i = lambda *t: torch.tensor(t, device=DEV, dtype=torch.int32)
    got = ops.attention_sink(q, k[0], v[0], i(0, 200), i(0, 330), i(130), [200], [130], 128 ** -0.5, sink)
    ok = torch.arange(330, device=DEV)[None] <= torch.arange(130, 330, device=DEV)[:, None]
    want, _, mag = reference(q[None], k, v, ok, 128 ** -0.5, sink)
    close(got[None], want, mag)
