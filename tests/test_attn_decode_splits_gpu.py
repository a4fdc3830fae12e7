"""One query a sequence: splits of one round of work-groups, for batches that divide the compute units and that do not, down to a single split."""
import pytest
import torch

from test_attention_two_waves_gpu import close, reference

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,G,gq,Lk", [(1, 8, 5, 1501), (3, 8, 5, 1501), (5, 8, 5, 700), (12, 8, 5, 1501), (20, 8, 4, 333), (32, 8, 1, 97), (33, 8, 2, 65), (3, 2, 20, 2500), (200, 2, 3, 31)])
def test_rounds(B, G, gq, Lk):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(B * Lk)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).bfloat16()
    q, k, v = r(B, 1, G * gq, 128), r(B, Lk, G, 128), r(B, Lk, G, 128)
    got, lse = ops.flash_attn_decode(q, k, v, return_lse=True)
    want, wlse, mag = reference(q, k, v, torch.ones(1, Lk, dtype=torch.bool, device=DEV), 128 ** -0.5)
    close(got, want, mag)
    assert (lse.double() - wlse).abs().max() <= 128 * 2.0 ** -24 * float(q.double().norm(dim=3).max() * k.double().norm(dim=3).max()) * 128 ** -0.5 + 2.0 ** -20
