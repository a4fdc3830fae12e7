"""The decode step's state update for several sequences: by every number of rows a wave, dense and with distances, against the sequences one at a time."""
import pytest
import torch

from timeviper_amd import kernels as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 10 and 20, 8 and 4 rows a wave at d_state 128; head dims that no number of rows divides go the one-sequence kernel's way
@pytest.mark.parametrize("B,H,P,G,N", [(2, 128, 80, 8, 128), (3, 128, 80, 8, 128), (4, 128, 80, 8, 128), (7, 128, 80, 8, 128), (2, 128, 64, 8, 128), (9, 128, 64, 1, 128), (2, 128, 68, 4, 128),
                                       (2, 128, 65, 8, 128), (5, 64, 80, 4, 64), (9, 128, 64, 2, 64), (2, 96, 40, 3, 256), (9, 64, 64, 2, 256), (40, 16, 64, 1, 128), (5, 128, 72, 8, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("wide", [False, True])
def test_sequences_together(B, H, P, G, N, dtype, wide):
    g = torch.Generator(device=DEV).manual_seed(B * H + P + N)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    cols = H * P + 2 * G * N + H
    row = r(B, cols + 24).to(dtype)
    x, Bm, Cm, dt = row[:, :cols].split([H * P, G * N, G * N, H], dim=1)
    if not wide:
        x, Bm, Cm, dt = (t.contiguous() for t in (x, Bm, Cm, dt))
    A, D, bias, state = -r(H).abs() - .1, r(H), r(H), r(B, H, P, N)
    step = lambda s, i: ops.selective_state_update(s, x[i].unflatten(1, (H, P)), dt[i], A, Bm[i].unflatten(1, (G, N)), Cm[i].unflatten(1, (G, N)), D, dt_bias=bias, dt_softplus=True)
    each = [state[b:b + 1].clone() for b in range(B)]
    want = torch.cat([step(s, slice(b, b + 1)) for b, s in enumerate(each)])
    guard = torch.full((B + 1, H, P, N), 7.0, device=DEV)
    guard[:B] = state
    got = step(guard[:B], slice(0, B))
    # the same operations in the same order
    assert torch.equal(got, want) and torch.equal(guard[:B], torch.cat(each)) and (guard[B] == 7).all()
