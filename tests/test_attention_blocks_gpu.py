"""How the flash kernel's work-groups are dealt out: query blocks of all heads by falling cost, and the sequences of a packed step in one launch."""
import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from timeviper_amd import kernels
    return kernels


def rnd(shape, seed):
    return torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).bfloat16()


def reference(q, k, v, scale, start, window=None, keep=0):
    """fp32 softmax attention of q (n, H, d) behind `start` earlier keys"""
    n, H, _ = q.shape
    k, v = (t.float().repeat_interleave(H // t.shape[1], 1).transpose(0, 1).contiguous() for t in (k, v))
    s = torch.bmm(q.float().transpose(0, 1).contiguous(), k.transpose(1, 2).contiguous()) * scale
    p = torch.arange(start, start + n, device=q.device)[:, None]
    j = torch.arange(k.shape[1], device=q.device)[None]
    see = j <= p
    if window is not None:
        see = see & ((p - j < window) | (j < keep))
    return torch.bmm(torch.softmax(s.masked_fill(~see, -math.inf), -1), v).transpose(0, 1)


def close(got, want):
    # bf16 weights and output: 2^-8 of the largest value a row mixes
    assert (got.float() - want).abs().max() <= 2.0 ** -7 * max(1.0, float(want.abs().max()))


# (batch x heads) pairs below, at and beside a multiple of the 8 XCDs; one, two and several query blocks
@pytest.mark.parametrize("B,H,G", [(1, 3, 1), (1, 8, 8), (2, 5, 5), (1, 28, 4), (3, 12, 4)])
@pytest.mark.parametrize("Lq,Lk", [(65, 65), (129, 400), (257, 257), (700, 700)])
def test_causal_blocks_of_all_heads(K, B, H, G, Lq, Lk):
    q, k, v = rnd((B, Lq, H, 128), 1), rnd((B, Lk, G, 128), 2), rnd((B, Lk, G, 128), 3)
    o = K.flash_attn_func(q, k, v, causal=True)
    for b in range(B):
        close(o[b], reference(q[b], k[b], v[b], 128 ** -0.5, Lk - Lq))


# more sequences than one launch takes; all short (128-row blocks); long and single-token ones together; portions behind earlier tokens
@pytest.mark.parametrize("counts,starts", [([1 + 7 * i % 53 for i in range(67)], [0] * 67), ([600, 1, 129, 300], [0, 0, 0, 0]),
                                           ([5, 260, 1, 40], [300, 17, 511, 0])])
@pytest.mark.parametrize("window,keep", [(64, 5), (1 << 30, 0)])
def test_packed_sequences_share_a_launch(K, counts, starts, window, keep):
    H, G, d, e = 6, 2, 64, 128
    n, cap = len(counts), max(a + c for a, c in zip(starts, counts)) + 3
    cache = rnd((n + 2, cap, G * (d + e)), 1)
    slots = [(5 * i + 1) % (n + 2) if math.gcd(5, n + 2) == 1 else i for i in range(n)]
    T = sum(counts)
    q, gate = rnd((T, H, d), 2), rnd((T, H, e), 3)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    cu = [0]
    for c in counts:
        cu.append(cu[-1] + c)
    plan = SimpleNamespace(slots=tuple(slots), counts=tuple(counts), starts=tuple(starts), cu=i32(cu), start=i32(starts), slot=i32(slots), decode=False,
                           seq=i32([b for b, c in enumerate(counts) for _ in range(c)]), rows=i32(list(range(T))), keys=None, moving=None)
    out = torch.full((T, H + 1, e), 9.0, device=DEV).bfloat16()
    o = K.attention_window(q, cache, plan, G, 0.11, window, keep, gate=gate, out=out[:, :H])
    assert o.data_ptr() == out.data_ptr() and (out[:, H] == 9).all()
    for s, a, c, r in zip(slots, starts, counts, cu):
        k, v = cache[s, :a + c].split([G * d, G * e], 1)
        want = reference(q[r:r + c], k.unflatten(1, (G, d)), v.unflatten(1, (G, e)), 0.11, a, window, keep)
        close(o[r:r + c], want * torch.sigmoid(gate[r:r + c].float()))


@pytest.mark.parametrize("causal", [False, True])
def test_more_query_blocks_than_a_grid_dimension(K, causal):
    """20 480 000 (batch, head) pairs of one query: a key of its own is all that each sees"""
    q, v = rnd((20000, 1, 1024, 8), 1), rnd((20000, 1, 1024, 8), 2)
    o, lse = K.flash_attn_func(q, q, v, causal=causal, return_lse=True)
    assert torch.equal(o, v)
    want = (q[:, 0].float() ** 2).sum(-1) * 8 ** -0.5
    assert (lse[:, :, 0] - want).abs().max() <= 1e-5 * want.abs().max()
