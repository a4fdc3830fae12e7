"""linear_fused where whole rounds of large tiles take the leading rows and small tiles the rest (kernels.lead_rows), against fp32."""
import pytest
import torch
import torch.nn.functional as F

DEV = "cuda"


# one row behind the lead, a whole small tile, one more, the most that the rule takes; 0: a full last round, too many small tiles, contractions and widths outside
@pytest.mark.parametrize("rows,n,k,gelu,lead", [(3841, 4352, 1152, True, 3840), (4374, 4352, 1152, True, 3840), (4640, 4352, 1152, True, 3840), (4750, 4352, 1152, True, 0),
                                                (3645, 4352, 1152, True, 0), (5103, 3456, 1152, False, 4608), (23552, 3456, 1152, False, 0), (23400, 3456, 1152, True, 23296),
                                                (729, 4352, 1152, True, 0), (4374, 4352, 4480, True, 0), (12000, 1152, 1152, True, 0)])
def test_rule(rows, n, k, gelu, lead):
    from timeviper_amd import kernels as K
    assert K.lead_rows(rows, n, k, K.GEMM_BIAS_GELU if gelu else K.GEMM_BIAS) == lead


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3841, 3968, 3969, 4374, 4640])
@pytest.mark.parametrize("gelu", [True, False])
@pytest.mark.parametrize("form", ["bias", "fp32 bias", "none", "rows"])
def test_against_fp32(rows, gelu, form):
    from timeviper_amd import kernels as K
    n, k = 4352, 1152
    epi = K.GEMM_BIAS_GELU if gelu else K.GEMM_BIAS
    assert K.lead_rows(rows, n, k, epi) == 3840
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, k + 64, generator=g, device=DEV).bfloat16()[:, :k] if form == "rows" else torch.randn(rows, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).bfloat16()
    b = None if form == "none" else torch.randn(n, generator=g, device=DEV)
    b = b.bfloat16() if form in ("bias", "rows") else b
    room = torch.full((rows + 1, n + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out = room[:rows, :n] if form == "rows" else None
    y = K.linear_fused(x, w, b, epi, out=out)
    want = F.linear(x.float(), w.float(), None if b is None else b.float())
    if gelu:
        want = F.gelu(want.bfloat16().float())
    # bf16 has 8 bits: the rounding of the sum s may fall to the other side of a tie, one step of at most 2^-7 |s|, which the GELU passes on times 1.13 at most
    # (below zero, where the result is small against s: times 0.13, of |s| < 4: 4e-3), and the result's own rounding is 2^-8 of it: 1.63 x 2^-7 in all
    err = (y.float() - want).abs()
    assert bool((err <= 1.63 * 2 ** -7 * want.abs() + 4.1e-3).all()), err.max()
    if form == "rows":
        assert bool((room[rows:] == 7).all()) and bool((room[:, n:] == 7).all())
