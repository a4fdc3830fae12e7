"""The products of a parallel layer's prompt with what stands behind them: gated pair, residual stream, token side."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def rand(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return lambda *s: torch.randn(s, generator=g, device=DEV)


# edges of tiles (256 rows, 128 outputs), one tile and more than one round of them, an even number of steps from four on
@pytest.mark.parametrize("M,N,K", [(256, 128, 256), (257, 136, 384), (511, 264, 512), (2100, 5632, 256)])
def test_gated_pair(M, N, K):
    from timeviper_amd import kernels as ops
    r = rand(M)
    x, w, b = r(M, K).to(BF), (K ** -0.5 * r(2 * N, K)).to(BF), r(2 * N).to(BF)
    wide = torch.full((M, N + 24), 7.0, device=DEV, dtype=BF)
    out = wide[:, 8:8 + N]
    ops.glu_linear(x, w, b, out)
    g, u = (x.double() @ w.double().T + b.double()).split(N, 1)
    want = F.gelu(g, approximate="tanh") * u
    # fp32 sums and functions (1e-5 of the factors; the slope of the activation is below 1.13) and one rounding
    bound = 2.0 ** -8 * want.abs() + 2e-5 * (g.abs() + 1) * (u.abs() + 1)
    assert ((out.double() - want).abs() <= bound).all()
    assert (wide[:, :8] == 7).all() and (wide[:, 8 + N:] == 7).all()


@pytest.mark.parametrize("M,N,K,splits", [(1, 4, 192, 1), (300, 516, 1088, 1), (255, 260, 640, 3), (513, 1024, 7680, 16)])
def test_onto_the_stream(M, N, K, splits):
    from timeviper_amd import kernels as ops
    r = rand(N)
    x, w, b, res = r(M, K).to(BF), (K ** -0.5 * r(N, K)).to(BF), r(N).to(BF), r(M, N)
    got, h = ops.split_add_linear(x, w, res, b, splits)
    want = res.double() + x.double() @ w.double().T + b.double()
    assert ((got.double() - want).abs() <= (x.double().abs() @ w.double().abs().T + want.abs() + 4) * K * 2.0 ** -24).all()
    assert torch.equal(h, got.to(BF))


# small tiles with a split contraction: edges of the three tiles, uneven splits, a step a split, more splits than one pass of the sum; slices, no bias
@pytest.mark.parametrize("M,N,K", [(1, 1024, 4096), (63, 1032, 4160), (65, 2048, 7680), (130, 1536, 5632), (300, 1032, 4224)])
@pytest.mark.parametrize("tile,splits", [(0, 3), (2, 1), (2, 11), (3, 8), (3, 64)])
def test_small_add(M, N, K, tile, splits):
    from timeviper_amd import kernels as ops
    r = rand(M + N)
    x, w, b, res = r(M, K + 8).to(BF)[:, :K], (K ** -0.5 * r(N, K + 8)).to(BF)[:, 8:], r(N).to(BF) if tile else None, r(M, N)
    got, h = ops.small_add_linear(x, w, res, b, tile, splits)
    want = res.double() + x.double() @ w.double().T + (0 if b is None else b.double())
    # fp32 sums (relative 2^-24 an addition, of the sum of magnitudes)
    assert ((got.double() - want).abs() <= (x.double().abs() @ w.double().abs().T + want.abs() + 4) * K * 2.0 ** -24).all()
    assert torch.equal(h, got.to(BF)) and torch.equal(got, ops.small_add_linear(x, w, res, b, tile, splits)[0])


def test_small_add_plan_of_long_contractions():
    from timeviper_amd import kernels as ops
    for rows, n, k, want in ((768, 1024, 16384, True), (769, 1024, 16384, False), (900, 1536, 10240, False), (1024, 1456, 8960, True)):
        assert (ops.small_add_plan(rows, n, k) is not None) == want


# W asked for ahead and not
@pytest.mark.parametrize("M", [287, 288])
@pytest.mark.parametrize("tile,splits", [(0, 2), (2, 3), (3, 8)])
def test_small_add_asks_ahead(M, tile, splits):
    """whole numbers: exact, whatever the order of the sums"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + splits)
    r = lambda *s: torch.randint(-3, 4, s, generator=g, device=DEV)
    x, w, res = r(M, 4160).to(BF), r(1032, 4160).to(BF), r(M, 1032).float()
    got, h = ops.small_add_linear(x, w, res, None, tile, splits)
    want = res.double() + x.double() @ w.double().T
    assert torch.equal(got.double(), want) and torch.equal(h, want.to(BF))


def test_small_add_plan():
    from timeviper_amd import kernels as ops
    for rows, n, k, want in ((17, 2048, 7680, True), (1024, 2048, 7680, True), (1025, 2048, 7680, False), (2048, 1024, 5120, True), (300, 3072, 11264, False), (300, 2048, 2048, False)):
        plan = ops.small_add_plan(rows, n, k)
        assert (plan is not None) == want
        if plan:
            tm, tn = {0: (128, 128), 2: (64, 128), 3: (64, 64)}[plan[0]]
            assert -(-rows // tm) * -(-n // tn) * plan[1] <= ops.CUS and k // 64 >= plan[1]
    z = lambda *s: torch.zeros(s, device=DEV, dtype=BF)
    for bad in ((z(4, 4096), z(1028, 4096)), (z(4, 4104), z(1024, 4104))):      # outputs no multiple of 8, contraction none of 64
        assert ops.small_add_takes(*bad) is None
        with pytest.raises(ops.TimeViperHipError):
            ops.small_add_linear(*bad, torch.zeros(4, bad[1].shape[0], device=DEV))


# tiles of 32 rows, units of 32 columns: fewer than the eight waves, no multiple of them; ids on both ends of the table, a slice of a wider one
@pytest.mark.parametrize("T,D", [(1, 32), (31, 96), (33, 288), (64, 2048), (515, 2080)])
def test_token_side(T, D):
    from timeviper_amd import kernels as ops
    r = rand(T)
    h, g, p, table = r(T, D + 8).to(BF)[:, :D], (D ** -0.5 * r(128, D)).to(BF), (128 ** -0.5 * r(D, 128)).to(BF), r(50, 384).to(BF)[:, 132:260]
    ids = torch.randint(0, 50, (T,), device=DEV)
    ids[0], ids[-1] = 0, 49
    got = ops.token_side(h, ids, table, g, p).double()
    s = h.double() @ g.double().T
    z = F.gelu(s, approximate="tanh") * table[ids].double()
    want = z @ p.double().T
    # roundings of the 128 sums, of z (2^-8 each, the first through a slope below 1.13) and of the result
    dz = (1.13 * 2.0 ** -8 * s.abs() + 1e-5) * table[ids].double().abs() + 2.0 ** -8 * z.abs()
    assert ((got - want).abs() <= 1.02 * dz @ p.double().abs().T + 2.0 ** -8 * want.abs()).all()
    ids[T // 2] = 50
    got, want[T // 2] = ops.token_side(h, ids, table, g, p), 0
    assert (got[T // 2] == 0).all()


def test_refused():
    from timeviper_amd import kernels as ops
    z = lambda *s: torch.zeros(s, device=DEV, dtype=BF)
    for x, w, n in ((z(255, 256), z(256, 256), 128), (z(256, 320), z(256, 320), 128), (z(256, 256), z(240, 256), 120)):
        with pytest.raises(ops.TimeViperHipError):
            ops.glu_linear(x, w, z(2 * n), z(x.shape[0], n))
    with pytest.raises(ops.TimeViperHipError):
        ops.token_side(z(4, 64), torch.zeros(4, dtype=torch.long, device=DEV), z(9, 64), z(64, 64), z(64, 64))
    with pytest.raises(ops.TimeViperHipError):
        ops.split_add_linear(z(4, 100), z(64, 100), torch.zeros(4, 64, device=DEV))


# few rows: several work-groups a block of rows, each with a share of the outputs (8, 6 that become 4, 2, one; a width of fewer, and of uneven, turns)
@pytest.mark.parametrize("D", [32, 288, 2048, 2080])
def test_token_side_shares(D):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(D)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    T = 6200
    h, table, gate, proj = r(T, D).bfloat16(), r(500, 128).bfloat16(), (r(128, D) * D ** -0.5).bfloat16(), (r(D, 128) * 128 ** -0.5).bfloat16()
    ids = torch.randint(0, 500, (T,), generator=g, device=DEV)
    whole = ops.token_side(h, ids, table, gate, proj)
    for n in (1, 31, 33, 700, 1000, 1600, 2900, 3100):
        assert torch.equal(ops.token_side(h[:n], ids[:n], table, gate, proj), whole[:n])      # a row's sums do not depend on the others


# both sides of each line
@pytest.mark.parametrize("rows,glu,add", [(255, False, 16), (512, False, 16), (700, True, 10), (1300, False, 5), (1800, True, 4), (4096, True, 2), (6011, True, 0)])
def test_rules(rows, glu, add):
    from timeviper_amd import kernels as ops
    h, u = torch.empty(rows, 2048, device=DEV, dtype=BF), torch.empty(rows, 7680, device=DEV, dtype=BF)
    inp, out = torch.empty(16384, 2048, device=DEV, dtype=BF)[5120:], torch.empty(2048, 7680, device=DEV, dtype=BF)
    with torch.no_grad():
        assert ops.glu_takes(h, inp) is glu and ops.split_add_takes(u, out) == add
        assert not ops.glu_takes(h[:, 4:], inp[:, 4:]) and not ops.split_add_takes(u[:, 4:], out[:, 4:])
    assert not ops.glu_takes(h, inp) and not ops.split_add_takes(u, out)       # gradients enabled


# a prompt on small tiles, one on the gated pair and on shared tiles, one on the library; biases that are slices of a larger tensor
@pytest.mark.parametrize("rows", [40, 700, 1400])
@pytest.mark.parametrize("off", [0, 1, 4])
def test_biases_at_any_address(rows, off):
    """a layer's biases off 16 bytes: the library's product, as for any other operand that the kernels do not read"""
    from timeviper_amd.model.llm.fogorax import FogoraxConfig, FogoraxForCausalLM
    mix = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1024, "keep_first": 64}}
    with torch.device("meta"):
        llm = FogoraxForCausalLM(FogoraxConfig(vocab_size=320, hidden_size=2048, side_dim=128, max_positions=2048,
                                               layers=[{"type": "attention", "mixer": mix, "mlp": {"kind": "dense", "ff": 5632}}]))
    llm = llm.to(BF).to_empty(device=DEV).requires_grad_(False)
    r = rand(5)
    for p in llm.parameters():
        p.copy_(0.02 * r(*p.shape))
    ids = torch.randint(0, 320, (rows,), generator=torch.Generator(device=DEV).manual_seed(rows), device=DEV)

    def logits():
        cache = llm.new_cache(1, capacity=rows)
        return llm.step(ids, cache, cache.plan(cache.default_slots, [rows]))
    with torch.inference_mode():
        want = logits()
        for layer in llm.backbone.layers:
            for name in ("inp_bias", "out_bias"):
                b = getattr(layer, name)
                moved = torch.empty(b.numel() + 8, device=DEV, dtype=BF)[off:off + b.numel()].copy_(b)
                assert moved.data_ptr() % 16 == 2 * off
                layer._parameters[name] = torch.nn.Parameter(moved, requires_grad=False)
        got = logits()
    # the same products with other roundings: gate and factor are rounded, the sum is rounded before it meets the stream
    assert torch.equal(got, want) if off == 0 else (got - want).norm() < 2.0 ** -6 * want.norm()


# a caller that does not wait for its launches: both sides of each line
@pytest.mark.parametrize("rows,D,ff,glu,add,side", [(300, 3072, 8192, False, 0, False), (400, 3072, 8192, False, 10, False), (700, 3072, 8192, True, 7, False), (203, 4096, 11008, False, 16, False),
                                                    (40, 4096, 11008, False, 0, False), (1400, 3072, 8192, False, 3, False), (1800, 2048, 5632, True, 4, False), (6011, 2048, 5632, True, 0, True),
                                                    (1800, 1024, 4096, True, 0, True), (6011, 4096, 11008, True, 0, True), (6011, 8192, 28672, False, 0, False)])
def test_rules_of_a_busy_device(rows, D, ff, glu, add, side):
    from timeviper_amd import kernels as ops
    z = lambda *s: torch.empty(s, device=DEV, dtype=BF)
    h, u, inp, out = z(rows, D), z(rows, D + ff), z(2 * ff, D), z(D, D + ff)
    with torch.no_grad():
        assert bool(ops.glu_takes(h, inp, None, False)) is glu and ops.split_add_takes(u, out, None, False) == add
        assert ops.side_takes(h, z(9, 128), z(128, D), z(D, 128), False) is side and ops.side_takes(h, z(9, 128), z(128, D), z(D, 128))


@pytest.mark.parametrize("rows,D,side", [(2048, 2048, False), (2049, 2048, True), (17, 1024, True), (5999, 4096, False)])
def test_rule_of_the_token_side(rows, D, side):
    from timeviper_amd import kernels as ops
    z = lambda *s: torch.empty(s, device=DEV, dtype=BF)
    with torch.no_grad():
        assert ops.side_takes(z(rows, D), z(9, 128), z(128, D), z(D, 128), False) is side
