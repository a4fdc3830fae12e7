"""linear_fused and glu_linear where whole rounds of large tiles take the leading rows and small tiles the rest (kernels.lead_rows, glu_lead), against fp32."""
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


# one small tile a compute unit, two on some, too many; a single large tile's rows missing, a full last round, less than a round
@pytest.mark.parametrize("rows,n,lead,tile", [(6011, 5632, 5888, 0), (3196, 5632, 2816, 1), (4750, 5632, 4750, -1), (1281, 5632, 1280, 0), (2048, 4096, 2048, -1), (1000, 5632, 1000, -1),
                                              (300, 40000, 300, -1)])
def test_pair_rule(rows, n, lead, tile):
    from timeviper_amd import kernels as K
    assert K.glu_lead(rows, n) == (lead, tile)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,tile", [(2049, 0), (2176, 0), (2177, 0), (2400, 0), (2600, 1)])
@pytest.mark.parametrize("sliced", [True, False])
def test_pair_against_fp64(rows, tile, sliced):
    from timeviper_amd import kernels as K
    n, k = 4096, 384
    assert K.glu_lead(rows, n) == (2048, tile)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn(rows, k + 64 * sliced, generator=g, device=DEV).bfloat16()[:, :k]
    w, b = (torch.randn(2 * n, k, generator=g, device=DEV) * k ** -0.5).bfloat16(), torch.randn(2 * n, generator=g, device=DEV).bfloat16()
    room = torch.full((rows + 1, n + 24), 7.0, dtype=torch.bfloat16, device=DEV)
    out = room[:rows, 8:8 + n]
    with torch.inference_mode():
        K.glu_linear(x, w, b, out)
    gate, up = (x.double() @ w.double().T + b.double()).split(n, 1)
    want = F.gelu(gate, approximate="tanh") * up
    # fp32 sums and functions (1e-5 of the factors; the slope of the activation is below 1.13) and one rounding
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * (gate.abs() + 1) * (up.abs() + 1)).all()
    assert (room[rows:] == 7).all() and (room[:, :8] == 7).all() and (room[:, 8 + n:] == 7).all()
