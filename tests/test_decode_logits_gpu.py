"""The logits of a decoded token as fp32 out of the product itself, the last norm in front of it, and the counters behind the greedy choice: the values of
the separate launches, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mk(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed + sum(shape)), device=DEV).bfloat16()


# rows of one work-group or less, a remainder of the waves, K that the matrix cores do not take (8, 4 488) or the split kernel does (8 192, 10 240)
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k,bias", [(1, 64, False), (1001, 4488, True), (9001, 4480, False), (513, 8, True), (20000, 8192, False), (7000, 10240, True)])
def test_logits(rows, n, k, bias):
    from timeviper_amd import kernels as K
    x, w, b = _mk(rows, 1, k), _mk(n, k, seed=1) * k ** -0.5, _mk(n, seed=2) if bias else None
    got = K.gemv_fused(x, w, b, out_dtype=torch.float32)
    want = K.gemv_fused(x, w, b).float()
    assert got.dtype == torch.float32 and got.shape == want.shape and torch.equal(got, want)


@pytest.mark.parametrize("n,k", [(9001, 4480), (100, 8), (4000, 8192), (513, 1032)])
@pytest.mark.parametrize("add", [True, False])
@pytest.mark.parametrize("nw", [torch.float32, torch.bfloat16])
def test_norm_in_front(n, k, add, nw):
    from timeviper_amd import kernels as K
    x, d, w, g = _mk(1, 1, k), _mk(1, 1, k, seed=3) if add else None, _mk(n, k, seed=1) * k ** -0.5, _mk(k, seed=4).to(nw)
    got = K.gemv_fused(x, w, None, K.GEMV_RMSNORM, delta=d, norm_weight=g, eps=1e-5, out_dtype=torch.float32)
    want = K.gemv_fused(x, w, None, K.GEMV_RMSNORM, delta=d, norm_weight=g, eps=1e-5).float()
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,n,k", [(2, 100, 64), (5, 9001, 4480), (17, 4099, 4480), (32, 515, 1024)])
def test_rows_rounded(rows, n, k):
    from timeviper_amd import kernels as K
    x, w, b = _mk(rows, k), _mk(n, k, seed=1) * k ** -0.5, _mk(n, seed=2)
    assert torch.equal(K.rows_linear(x, w, b, out_dtype=torch.float32, rounded=True), K.rows_linear(x, w, b).float())


@pytest.mark.parametrize("rows,n", [(1, 8192), (5, 131072), (3, 100), (2, 8195)])
@pytest.mark.parametrize("lens", [1, 64, 70])
def test_counters(rows, n, lens):
    from timeviper_amd import kernels as K
    x = torch.randn(rows, n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV)
    p, c = torch.tensor([41], device=DEV), torch.arange(lens, dtype=torch.int32, device=DEV)
    want = c + 1
    assert torch.equal(K.argmax_rows(x, (p, c)), x.argmax(-1)) and torch.equal(c, want) and p.item() == 42


def test_a_cache_that_counts_otherwise_is_asked():
    from timeviper_amd.model.llm.nano import HybridMambaAttentionDynamicCache as Cache

    class Other(Cache):
        def advance_static_device(self):
            raise AssertionError("not called here")
    pair = (torch.zeros(1, dtype=torch.int64), torch.zeros(2, dtype=torch.int32))
    for cls, want in ((Cache, pair), (Other, None)):
        c = cls.__new__(cls)
        c._static = {3: pair}
        assert c.static_counters() is want
        c._static = {3: pair, 4: pair}
        assert c.static_counters() is None
