"""The causal convolution's strips (csrc/conv1d.hip) at their edges, in both ways it loads its weights, against float64."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(x, w, b, halo, silu):
    K = w.shape[1]
    left = torch.zeros_like(x[:, :K - 1]) if x.shape[1] >= K - 1 else x.new_zeros(x.shape[0], K - 1, x.shape[2])
    full = torch.cat([left if halo is None else halo, x], 1).double()
    y = sum(full[:, j:j + x.shape[1]] * w[:, j].double() for j in range(K)) + (0 if b is None else b.double())
    return F.silu(y) if silu else y


# strips of 8 tokens, runs of strips on 8 XCDs (64 tokens), chunks of 64; channels that end inside a block; weights and bias of any alignment
@pytest.mark.parametrize("L", [1, 7, 8, 9, 63, 65, 200])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,shift,halo", [(4, 0, True), (4, 1, False), (3, 0, False), (2, 3, True)])
def test_strips(L, dtype, K, shift, halo):
    from timeviper_amd import kernels as ops
    B, di, G, N = 2, 2064, 2, 128
    C = di + 2 * G * N
    g = torch.Generator(device=DEV).manual_seed(L * 8 + K)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(dtype)
    x = r(B, L, C + 32)[..., 16:16 + C]
    w, b = r(C * K + shift)[shift:].view(C, K), r(C + shift)[shift:]
    h = r(B, K - 1, C) if halo else None
    want = reference(x, w, b, h, True)
    # fp32 accumulation: K + 1 rounded terms and the SiLU's two instructions of 1 ulp; one rounding to the output's type
    tol = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[dtype]
    bound = tol * (want.abs() + reference(x.abs(), w.abs(), b.abs(), None if h is None else h.abs(), False) * 2.0 ** -2 + 1e-6)
    xs, Bm, Cm, *cb = ops.causal_conv1d_xbc(x, w, b, di, G, N, activation="silu", halo=h, return_cb=True)
    got = torch.cat([xs, Bm.reshape(B, L, G * N), Cm.reshape(B, L, G * N)], -1)
    assert ((got.double() - want).abs() <= bound).all()
    if dtype is torch.bfloat16:                                # the other launch: no C.B^T, all channels in strips
        again = ops.causal_conv1d_xbc(x, w, b, di, G, N, activation="silu", halo=h)
        assert all(torch.equal(p, q) for p, q in zip(again, (xs, Bm, Cm)))
    if not halo:
        for act in (None, "silu"):
            want = reference(x, w, b, None, act == "silu")
            got = ops.causal_conv1d_fn(x.transpose(1, 2), w, b, activation=act).transpose(1, 2)
            assert ((got.double() - want).abs() <= bound + tol * want.abs()).all()
