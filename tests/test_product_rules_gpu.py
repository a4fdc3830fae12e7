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
