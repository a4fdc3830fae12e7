"""The scan of short sequences (csrc/ssd_cols.hip: column slices, no segments) against the token recurrence in 64 bits, over its modes."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def K():
    from timeviper_amd import kernels
    return kernels


def recurrence(x, dt, A, B, C, D, S, heads_of):
    """one sequence, token by token: x (L, H, P), dt (L, H) discretised, B / C (L, G, N), S (H, P, N); all fp64.  Outputs, final state, and the
    sums of the magnitudes of their terms"""
    y, ym, Sm = torch.empty_like(x), torch.empty_like(x), S.abs()
    for t in range(x.shape[0]):
        b, c, e = B[t, heads_of], C[t, heads_of], torch.exp(dt[t] * A)[:, None, None]
        new = (dt[t, :, None] * x[t])[:, :, None] * b[:, None]
        S, Sm = e * S + new, e * Sm + new.abs()
        y[t] = (S * c[:, None]).sum(-1) + D[:, None] * x[t]
        ym[t] = (Sm * c[:, None].abs()).sum(-1) + (D[:, None] * x[t]).abs()
    return y, S, ym, Sm


# chunk edges, one token, the last chunk nearly empty / nearly full; head dims of one to five slices; a group's slices spread over
# several heads; dt_std moves heads through floating, re-based, reset and standard steps
@pytest.mark.parametrize("L", [1, 63, 64, 65, 129, 200, 390])
@pytest.mark.parametrize("B,H,P,G,group_map", [(1, 8, 80, 2, "block"), (2, 8, 80, 2, "tile"), (1, 4, 32, 1, "block"), (1, 8, 64, 4, "block")])
@pytest.mark.parametrize("decay", ["slow", "mixed", "fast"])
def test_short_scan(K, L, B, H, P, G, group_map, decay):
    N = 128
    g = torch.Generator(device=DEV).manual_seed(L * 7 + H)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    proj = (1.3 * r(B, L, H * P + 16)).bfloat16()              # x and dt as slices of a wider row
    x, dt = proj[..., :H * P].unflatten(-1, (H, P)), proj[..., H * P + 2:H * P + 2 + H]
    bc = (0.3 * r(B, 2 * G, L, N)).bfloat16()
    Bm, Cm = bc[:, :G].transpose(1, 2), bc[:, G:].transpose(1, 2)
    A = -{"slow": torch.linspace(0.01, 1, H, device=DEV), "mixed": torch.linspace(0.01, 16, H, device=DEV),
          "fast": torch.linspace(8, 60, H, device=DEV)}[decay]
    bias, D = torch.linspace(-6, -1, H, device=DEV), r(H)
    init = r(B, H, P, N)
    y, fin, dec = K.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=True,
                                              group_map=group_map, return_total_decay=True)
    assert K.ssd_scan_last_kernel() == 9
    h = torch.arange(H, device=DEV)
    of = h % G if group_map == "tile" else h // (H // G)
    for b in range(B):
        d = F.softplus(dt[b].double() + bias.double())
        yr, Sr, ym, Sm = recurrence(x[b].double(), d, A.double(), Bm[b].double(), Cm[b].double(), D.double(), init[b].double(), of)
        # element by element: a term of y meets two bf16 operands that were rounded (x~ and C.B^T, or x~ inside the state and the state's copy:
        # 2^-8 each), a term of the state one, y is rounded itself (2^-8); 5 % for fp32 sums and exponents (differences of prefix sums)
        assert ((y[b].double() - yr).abs() <= 1.05 * (2.0 ** -7 * ym + 2.0 ** -8 * yr.abs()) + 1e-30).all()
        assert ((fin[b].double() - Sr).abs() <= 1.05 * 2.0 ** -8 * Sm + 1e-30).all()
        assert torch.allclose(dec[b].double(), (d * A.double()).sum(0), rtol=1e-4, atol=1e-4)


# slices up to 7 chunks, 9 at head dim 80 and 24 of more than 128 heads; heads in segments from there on; those up to 24 chunks a segment (here one: 512 heads), the march beyond
@pytest.mark.parametrize("B,H,P,G,chunks,kernels", [(1, 16, 64, 2, 8, (9, 10)), (1, 16, 80, 2, 10, (9, 10)), (1, 160, 80, 8, 25, (9, 10)), (1, 160, 32, 8, 8, (9, 10)),
                                                    (4, 128, 80, 8, 25, (10, 6))])
def test_either_side_of_a_line_agrees(K, B, H, P, G, chunks, kernels):
    N = 128
    g = torch.Generator(device=DEV).manual_seed(3)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    L = chunks * 64
    x, dt, Bm, Cm = r(B, L, H, P).bfloat16(), r(B, L, H).bfloat16(), (0.3 * r(B, L, G, N)).bfloat16(), (0.3 * r(B, L, G, N)).bfloat16()
    A, bias, D = -torch.linspace(0.02, 16, H, device=DEV), torch.full((H,), -4.0, device=DEV), r(H)

    def f(n):
        y, S = K.mamba_chunk_scan_combined(x[:, :n], dt[:, :n], A, Bm[:, :n], Cm[:, :n], D=D, dt_bias=bias, dt_softplus=True, return_final_states=True)
        return y, S, K.ssd_scan_last_kernel()
    (long, _, b), (short, fin, a) = f(L), f(L - 64)
    assert (a, b) == kernels
    K.ssd_scan_set_impl(6)
    try:
        march, Sm, six = f(L - 64)
    finally:
        K.ssd_scan_set_impl(0)
    assert six == 6
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    # (x~ is rounded to bf16 in another frame on each side, 2^-9 at most each)
    assert rel(long[:, :L - 64], short) < 5e-3 and rel(march, short) < 5e-3 and rel(Sm, fin) < 5e-3


def test_segments_that_rounding_up_leaves_without_chunks(K, monkeypatch):
    """64 heads, 120 chunks: sixteen segments of eight chunks are fifteen, and the sixteenth has nothing to read"""
    H, P, G, N, L = 64, 80, 8, 128, 120 * 64 - 5
    g = torch.Generator(device=DEV).manual_seed(5)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, dt, Bm, Cm = r(1, L, H, P).bfloat16(), r(1, L, H).bfloat16(), (0.3 * r(1, L, G, N)).bfloat16(), (0.3 * r(1, L, G, N)).bfloat16()
    A, bias, D, init = -torch.linspace(0.02, 16, H, device=DEV), torch.full((H,), -4.0, device=DEV), r(H), r(1, H, P, N)
    f = lambda: K.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=True)
    K.ssd_scan_set_impl(6)
    try:
        y, fin = f()
        assert K.ssd_scan_last_kernel() == 6
    finally:
        K.ssd_scan_set_impl(0)
    monkeypatch.setenv("TV_SSD_NSEG", "1")                     # (asks for the march by itself)
    y1, fin1 = f()
    assert K.ssd_scan_last_kernel() == 6 and not torch.equal(y, y1)
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    # x~ is rounded to bf16 in another frame on each side (2^-8 each), the carried-in states enter y as a product of their own
    assert torch.isfinite(y).all() and rel(y, y1) < 2.0 ** -7 and rel(fin, fin1) < 2.0 ** -7


@pytest.mark.parametrize("L", [1, 63, 64, 150])
@pytest.mark.parametrize("which", ["x", "B", "C"])
def test_operands_expanded_over_the_tokens(K, L, which):
    """rows that lie on top of each other: copied row by row below 64 tokens, the general recurrence from there on (one token has no distance)"""
    H, P, G, N = 8, 80, 2, 128
    g = torch.Generator(device=DEV).manual_seed(L)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).bfloat16()
    ops = {"x": r(1, L, H, P), "B": 0.3 * r(1, L, G, N), "C": 0.3 * r(1, L, G, N)}
    ops[which] = ops[which][:, :1].expand(-1, L, -1, -1)
    assert L == 1 or ops[which].stride(1) == 0
    x, Bm, Cm = ops.values()
    dt, A, bias, D = r(1, L, H), -torch.linspace(0.01, 16, H, device=DEV), torch.full((H,), -4.0, device=DEV), torch.ones(H, device=DEV)
    y, fin = K.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, return_final_states=True)
    assert K.ssd_scan_last_kernel() == (9 if L < 64 else 1)
    yr, Sr, ym, Sm = recurrence(x[0].double(), F.softplus(dt[0].double() + bias.double()), A.double(), Bm[0].double(), Cm[0].double(), D.double(),
                                torch.zeros(H, P, N, dtype=torch.float64, device=DEV), torch.arange(H, device=DEV) // (H // G))
    assert ((y[0].double() - yr).abs() <= 1.05 * (2.0 ** -7 * ym + 2.0 ** -8 * yr.abs()) + 1e-30).all()       # (as above)
    assert ((fin[0].double() - Sr).abs() <= 1.05 * 2.0 ** -8 * Sm + 1e-30).all()


# csrc/ssd_par.hip: a head per work-group, segments that start from the state their predecessors leave.  Chunk and segment edges, one segment (many heads, or slices
# that column work-groups cannot take), head dims with and without a single tile; decays that take a chunk as it is, raised, or with the true mask
@pytest.mark.parametrize("B,H,P,G,group_map,L", [
    (1, 8, 80, 2, "block", 640), (1, 8, 80, 2, "tile", 577), (2, 8, 80, 2, "block", 1089), (1, 4, 32, 1, "block", 705), (2, 8, 64, 4, "tile", 640),
    (1, 2, 80, 2, "block", 1), (1, 2, 80, 2, "block", 63), (1, 2, 80, 2, "tile", 130), (1, 6, 64, 2, "block", 513),
    (3, 128, 80, 8, "block", 65), (2, 128, 32, 8, "block", 500)])
@pytest.mark.parametrize("decay", ["slow", "mixed", "fast"])
def test_heads_in_segments(K, B, H, P, G, group_map, L, decay):
    N = 128
    g = torch.Generator(device=DEV).manual_seed(L * 7 + H)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    proj = (1.3 * r(B, L, H * P + H + 16 - H % 8)).bfloat16()  # x and dt as slices of a wider row
    proj = proj[..., :proj.shape[-1] // 8 * 8].contiguous()
    x, dt = proj[..., :H * P].unflatten(-1, (H, P)), proj[..., H * P:H * P + H]
    bc = (0.3 * r(B, 2 * G, L, N)).bfloat16()
    Bm, Cm = bc[:, :G].transpose(1, 2), bc[:, G:].transpose(1, 2)
    A = -{"slow": torch.linspace(0.01, 1, H, device=DEV), "mixed": torch.linspace(0.01, 16, H, device=DEV),
          "fast": torch.linspace(8, 60, H, device=DEV)}[decay]
    bias, D = torch.linspace(-6, -1, H, device=DEV), r(H)
    init = r(B, H, P, N)
    y, fin, dec = K.mamba_chunk_scan_combined(x, dt, A, Bm, Cm, D=D, dt_bias=bias, dt_softplus=True, initial_states=init, return_final_states=True,
                                              group_map=group_map, return_total_decay=True)
    assert K.ssd_scan_last_kernel() == 10
    h = torch.arange(H, device=DEV)
    of = h % G if group_map == "tile" else h // (H // G)
    for b in range(B):
        d = F.softplus(dt[b].double() + bias.double())
        yr, Sr, ym, Sm = recurrence(x[b].double(), d, A.double(), Bm[b].double(), Cm[b].double(), D.double(), init[b].double(), of)
        assert ((y[b].double() - yr).abs() <= 1.05 * (2.0 ** -7 * ym + 2.0 ** -8 * yr.abs()) + 1e-30).all()       # (as above)
        assert ((fin[b].double() - Sr).abs() <= 1.05 * 2.0 ** -8 * Sm + 1e-30).all()
        assert torch.allclose(dec[b].double(), (d * A.double()).sum(0), rtol=1e-4, atol=1e-4)
