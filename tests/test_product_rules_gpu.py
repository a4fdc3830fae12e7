"""Which kernel a product of the hybrid stack runs on, and what keeps it on torch.nn.Linear."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def linear(K, N, seed=0):
    with torch.device("meta"):
        lin = torch.nn.Linear(K, N, bias=False, dtype=BF)
    lin = lin.to_empty(device=DEV).requires_grad_(False)
    lin.weight.normal_(0, K ** -0.5, generator=torch.Generator(device=DEV).manual_seed(seed))
    return lin


@pytest.mark.parametrize("K,N,relu2", [(4480, 15680, True), (4480, 22656, False)])
def test_persistent_kernel_switched_off(K, N, relu2):
    """`gemm_set_persist(0)` (TV_GEMM_PERSIST=0): a long prompt's products are the library's, the squared ReLU among them"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    lin, x = linear(K, N), torch.randn(1, 2048, K, device=DEV).to(BF)
    with torch.no_grad():
        assert ops.large_takes(x, lin.weight, relu2)
        ops.gemm_set_persist(0)
        try:
            assert not ops.large_takes(x, lin.weight, relu2)
            got = nano._prompt_linear(lin, x, relu2)
        finally:
            ops.gemm_set_persist(-1)
        want = lin(x)
        assert torch.equal(got, ops.relu2(want, inplace=True) if relu2 else want)


# shared tiles, tiles of an odd number of steps, shared last rounds (which `large_takes` has too, or not), the squared ReLU of a single round
@pytest.mark.parametrize("K,N,relu2,rows", [(15680, 4480, False, 512), (15680, 4480, False, 3000), (4480, 22656, False, 2200), (10240, 4480, False, 8192),
                                            (4480, 15680, True, 700)])
def test_shared_tiles_switched_off(K, N, relu2, rows):
    """the same switch: the products that the split kernel has are the library's as well, and do not take the place of those that the persistent one gave up"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    lin, x = linear(K, N), torch.randn(1, rows, K, device=DEV).to(BF)
    with torch.no_grad():
        assert ops.split_takes(x, lin.weight, relu2) or ops.large_takes(x, lin.weight, relu2)
        ops.gemm_set_persist(0)
        try:
            assert ops.split_takes(x, lin.weight, relu2) is None
            got = nano._prompt_linear(lin, x, relu2)
        finally:
            ops.gemm_set_persist(-1)
        want = lin(x)
        assert torch.equal(got, ops.relu2(want, inplace=True) if relu2 else want)


def test_gated_pair_switched_off():
    from timeviper_amd import kernels as ops
    h, w = torch.empty(6011, 2048, device=DEV, dtype=BF), torch.empty(2 * 5632, 2048, device=DEV, dtype=BF)
    with torch.no_grad():
        assert ops.glu_takes(h, w)
        ops.gemm_set_persist(0)
        try:
            assert not ops.glu_takes(h, w)
        finally:
            ops.gemm_set_persist(-1)


@pytest.mark.parametrize("rows", [5, 32])
def test_output_layer_keeps_its_gradient(rows):
    """logits of 5..32 rows of a packed model: differentiable in the table where gradients are enabled"""
    from timeviper_amd.model.llm.packed import vocabulary_logits
    h = torch.randn(rows, 128, device=DEV).to(BF)
    table = torch.nn.Parameter(torch.randn(300, 128, device=DEV).to(BF))
    up = torch.randn(rows, 300, device=DEV).to(BF).float()
    vocabulary_logits(h, table).backward(up)
    want = up.double().T @ h.double()                               # fp32 sums of `rows` products, rounded to bf16
    assert (table.grad.double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    with torch.no_grad():
        got = vocabulary_logits(h, table)
    assert got.dtype == torch.float32 and (got.double() - h.double() @ table.double().T).abs().max() < 1e-3


# (4 480 wide stack: in_proj, out_proj, up_proj + squared ReLU) x rows on either side of each line
@pytest.mark.parametrize("N,K,relu2,rows,own", [(22656, 4480, False, 10007, True), (22656, 4480, False, 14000, False), (22656, 4480, False, 163940, False),
                                                (4480, 10240, False, 28000, True), (4480, 10240, False, 40000, False), (4480, 10240, False, 163940, False),
                                                (15680, 4480, True, 163940, True), (15680, 4480, False, 10007, False)])
def test_large_rule(N, K, relu2, rows, own):
    from timeviper_amd import kernels as ops
    x, w = torch.empty(1, rows, K, device=DEV, dtype=BF), torch.empty(N, K, device=DEV, dtype=BF)
    assert ops.large_takes(x, w, relu2) is own


@pytest.mark.parametrize("M", [1, 2, 4])
def test_decode_products_refuse_and_take_what_one_row_does(M):
    """gemv_fused: rows off their alignment, a convolution behind 8 192 inputs and groups of more than 2 048 channels are refused whatever the
    number of rows; a norm weight at an 8-byte address is taken"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(BF)
    w = r(96, 8192)
    with pytest.raises(ops.TimeViperHipError):
        ops.gemv_fused(r(M, 8192 + 8)[:, 4:-4], w)
    with pytest.raises(ops.TimeViperHipError):
        ops.gemv_fused(r(M, 8192), w, conv=(r(M, 32, 4), r(32, 4), None, 16))
    with pytest.raises(ops.TimeViperHipError):
        ops.gemv_fused(r(M, 8192), w, prologue=ops.GEMV_GATED, gate=r(M, 8192), norm_weight=r(8192), group_size=4096, eps=1e-5)
    x, nw = r(M, 512), 1 + 0.1 * r(516)
    off = nw[4:]
    assert off.data_ptr() % 16 == 8
    w = r(96, 512)
    got = ops.gemv_fused(x, w, prologue=ops.GEMV_RMSNORM, norm_weight=off, eps=1e-5)
    f = (x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-5) * off.double())
    want = f @ w.double().T
    # two roundings of the 512 normed values (2^-8 each, at random signs) and one of the sum
    bound = 2.0 ** -7 * torch.sqrt(f.square() @ w.double().square().T) * 2 + 2.0 ** -8 * want.abs()
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M,N,K,normed,rows", [(2, 1024, 1024, True, False), (2, 1024, 1024, False, True), (3, 1024, 1024, True, True), (2, 4096, 1024, True, True),
                                               (2, 4480, 4480, True, True), (1, 4480, 4480, True, False)])
def test_two_rows_of_a_small_matrix_are_one_launch(M, N, K, normed, rows, monkeypatch):
    from timeviper_amd import kernels as ops
    calls, real = [], ops._rows_product
    monkeypatch.setattr(ops, "_rows_product", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    x, w = torch.randn(M, K, device=DEV).to(BF), torch.randn(N, K, device=DEV).to(BF)
    kw = dict(prologue=ops.GEMV_RMSNORM, norm_weight=torch.ones(K, device=DEV), eps=1e-5) if normed else {}
    got = ops.gemv_fused(x, w, **kw)
    f = ops.rms_norm(x, torch.ones(K, device=DEV), 1e-5) if normed else x
    want = f.double() @ w.double().T
    assert bool(calls) is rows and ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + (f.double().abs() @ w.double().abs().T) * K * 2.0 ** -24).all()


@pytest.mark.parametrize("rows,N,K,own", [(17, 131072, 1024, True), (24, 131072, 1024, False), (32, 32768, 1024, True), (20, 131072, 1024, True)])
def test_output_layer_of_many_sequences(rows, N, K, own, monkeypatch):
    """more than 20 rows of the largest matrices are the library's: a step's output layer, and a packed model's"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    from timeviper_amd.model.llm.packed import vocabulary_logits
    lin, x = linear(K, N), torch.randn(rows, 1, K, device=DEV).to(BF)
    calls, real = [], ops.rows_linear
    monkeypatch.setattr(ops, "rows_linear", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    want = x[:, 0, :].double() @ lin.weight[-500:].double().T
    with torch.no_grad():
        for got in (nano._linear(lin, x)[:, 0], vocabulary_logits(x[:, 0], lin.weight)):
            assert (got[:, -500:].double() - want).abs().max() <= 2.0 ** -8 * want.abs().max()
    assert len(calls) == (2 if own else 0)


# both sides of each line of the short-prompt rule
@pytest.mark.parametrize("N,K,relu2,rows,own", [(22656, 4480, False, 64, True), (22656, 4480, False, 65, False), (4096, 4096, False, 48, False),
                                                (12288, 4096, False, 64, False), (12288, 4096, True, 64, True), (2048, 4096, False, 64, True), (2048, 4096, False, 96, False),
                                                (2048, 4096, True, 256, False), (4480, 5120, False, 256, True), (15680, 4480, True, 96, True),
                                                (4480, 15680, False, 203, True), (6144, 2048, False, 40, False)])
def test_short_prompt_rule(N, K, relu2, rows, own):
    from timeviper_amd import kernels as ops
    assert ops.mid_takes(torch.empty(1, rows, K, device=DEV, dtype=BF), torch.empty(N, K, device=DEV, dtype=BF), relu2) is own
