"""Products on small tiles (tv_gemm_small_fwd): edges of the three tiles, one to many stages of 64 columns, every epilogue; where they replace the library's."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (63, 72, 128), (65, 64, 192), (128, 128, 256), (129, 136, 320), (300, 264, 1152)])
def test_against_64_bits(M, N, K, tile):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + K)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, b, c = r(M, K + 16).to(BF)[:, 8:8 + K], (K ** -0.5 * r(N, K)).to(BF), r(N), r(M, N).to(BF)
    s = x.double() @ w.double().T
    sums = (x.double().abs() @ w.double().abs().T + 4) * K * 2.0 ** -24       # fp32 sums in any order
    one = lambda v, e: e + 2.0 ** -8 * (v.abs() + e)                           # ... and one rounding
    for bias in (None, b, b.to(BF)):
        want = s if bias is None else s + bias.double()
        got = ops.small_linear(x, w, bias, tile=tile).double()
        assert ((got - want).abs() <= one(want, sums)).all()
        got = ops.small_linear(x, w, bias, ops.GEMM_BIAS_GELU, tile=tile).double()
        want, e = F.gelu(want), 1.13 * one(want, sums) + 1e-6                 # the GELU of the rounded sum: its slope is below 1.13
        assert ((got - want).abs() <= one(want, e)).all()
    wide = torch.full((M, N + 16), 7.0, device=DEV, dtype=BF)
    out = wide[:, 8:8 + N]
    out.copy_(c)
    ops.small_linear(x, w, None, ops.GEMM_ACCUM, out=out, tile=tile)
    assert ((out.double() - (s + c.double())).abs() <= one(s + c.double(), sums)).all() and (wide[:, :8] == 7).all() and (wide[:, 8 + N:] == 7).all()
    w2, b2 = (K ** -0.5 * r(2 * N, K)).to(BF), r(2 * N).to(BF)
    f, u = (x.double() @ w2.double().T + b2.double()).split(N, 1)
    want = F.gelu(f, approximate="tanh") * u
    got = ops.small_linear(x, w2, b2, ops.GEMM_GLU, tile=tile).double()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * (f.abs() + 1) * (u.abs() + 1)).all()


@pytest.mark.parametrize("tile", [0, 1, 2, 3])
@pytest.mark.parametrize("stages", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13])
def test_every_end_of_the_ring(stages, tile):
    """whole numbers: exact, whatever the order of the sums; a number of stages that a slot, a wait or the parity of the fragments could miss"""
    from timeviper_amd import kernels as ops
    K = 64 * stages
    g = torch.Generator(device=DEV).manual_seed(K)
    r = lambda *s: torch.randint(-3, 4, s, generator=g, device=DEV).to(BF)
    x, w, c = r(193, K), r(200, K), r(193, 200)
    want = x.double() @ w.double().T + c.double()
    out = c.clone()
    ops.small_linear(x, w, None, ops.GEMM_ACCUM, out=out, tile=tile)
    assert torch.equal(out, want.to(BF))


# W asked for ahead and not: both sides of each line in rows and columns
@pytest.mark.parametrize("M,N,K,tile", [(191, 200, 3072, 3), (192, 200, 3072, 3), (193, 1032, 3136, 2), (320, 264, 3008, 0), (320, 264, 3072, 0), (191, 264, 1024, 1), (192, 264, 960, 1), (200, 264, 1024, 1),
                                        (511, 136, 1088, 1), (513, 136, 1088, 1)])
def test_weights_asked_for_ahead(M, N, K, tile):
    """whole numbers: exact, whatever the order of the sums"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + K)
    r = lambda *s: torch.randint(-3, 4, s, generator=g, device=DEV).to(BF)
    x, w = r(M, K), r(2 * N, K + 8)[:, :K]                     # (rows of W apart: the lines asked for are those of its rows)
    want = x.double() @ w.double().T
    assert torch.equal(ops.small_linear(x, w, tile=tile), want.to(BF))
    f, u = want.split(N, 1)
    got = ops.small_linear(x, w, torch.zeros(2 * N, device=DEV, dtype=BF), ops.GEMM_GLU, tile=tile).double()
    glu = F.gelu(f, approximate="tanh") * u
    assert ((got - glu).abs() <= 2.0 ** -8 * glu.abs() + 2e-5 * (f.abs() + 1) * (u.abs() + 1)).all()


@pytest.mark.parametrize("M,N,tile", [(1024, 1152, 3), (960, 1088, 3), (729, 3456, 2), (1025, 2048, 2), (2048, 4096, 3)])
def test_more_work_groups_than_a_round(M, N, tile):
    """a tile that gives way to the next larger one, and those that just do not"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M)
    r = lambda *s: torch.randint(-3, 4, s, generator=g, device=DEV).to(BF)
    x, w = r(M, 192), r(N, 192)
    assert torch.equal(ops.small_linear(x, w, None, tile=tile), (x.double() @ w.double().T).to(BF))


@pytest.mark.parametrize("rows,n,k,takes", [(2177, 1152, 1152, True), (2176, 1152, 1152, False), (1921, 1152, 4352, True), (1920, 1152, 4352, False), (3584, 1152, 4352, True),
                                            (3585, 1152, 4352, False), (2916, 1152, 6208, False), (2916, 1152, 960, False), (2916, 1148, 1152, False), (513, 4096, 2048, True), (512, 4096, 2048, False)])
def test_rule_of_a_full_round(rows, n, k, takes):
    from timeviper_amd import kernels as ops
    x, w = torch.empty(rows, k, device=DEV, dtype=BF), torch.empty(n, k, device=DEV, dtype=BF)
    assert not ops.round_takes(x, w)                                          # gradients enabled
    with torch.no_grad():
        assert ops.round_takes(x, w) == takes and not ops.round_takes(x[:, 4:], w[:, 4:]) and not ops.round_takes(x.float(), w.float())


@pytest.mark.parametrize("rows,n,k,takes", [(3584, 768, 3072, False), (3585, 768, 3072, True), (384, 6144, 4096, False), (640, 6144, 2752, True), (640, 6144, 2816, False), (1024, 2816, 2816, True)])
def test_rule_of_wide_and_narrow_outputs(rows, n, k, takes):
    from timeviper_amd import kernels as ops
    with torch.no_grad():
        assert ops.round_takes(torch.empty(rows, k, device=DEV, dtype=BF), torch.empty(n, k, device=DEV, dtype=BF)) is takes


def test_refused():
    from timeviper_amd import kernels as ops
    z = lambda *s: torch.zeros(s, device=DEV, dtype=BF)
    for x, w, kw in ((z(9, 96), z(64, 96), {}), (z(9, 64), z(60, 64), {}), (z(9, 68)[:, 4:], z(64, 64), {}), (z(9, 64), z(64, 64), dict(epilogue=ops.GEMM_ACCUM)),
                     (z(9, 64), z(64, 64), dict(epilogue=ops.GEMM_GLU)), (z(9, 64), z(64, 64), dict(tile=4)), (z(9, 64), z(64, 64), dict(epilogue=3))):
        with pytest.raises(ops.TimeViperHipError):
            ops.small_linear(x, w, **kw)


# rows x outputs x columns: both sides of each line
@pytest.mark.parametrize("rows,n,k,glu,tile", [(1, 1152, 1152, False, -1), (2, 1152, 1152, False, 3), (729, 1152, 1152, False, 3), (1458, 1152, 1152, False, 2), (729, 3456, 1152, False, 2),
                                               (1458, 3456, 1152, False, 1), (2304, 3456, 1152, False, 1), (2305, 3456, 1152, False, -1), (2187, 4352, 1152, False, -1),
                                               (1458, 1152, 4352, False, 3), (2187, 1152, 4352, False, -1), (729, 1152, 8192, False, -1), (200, 5632, 2048, True, 0),
                                               (512, 5632, 2048, True, 1), (700, 5632, 2048, True, -1), (729, 504, 1152, False, -1), (729, 1152, 1120, False, -1)])
def test_rule(rows, n, k, glu, tile):
    from timeviper_amd import kernels as ops
    x, w = torch.empty(rows, k, device=DEV, dtype=BF), torch.empty(n * (2 if glu else 1), k, device=DEV, dtype=BF)
    assert ops.small_tile(rows, n, k, glu) == tile and ops.small_takes(x, w, glu) == -1       # gradients enabled
    with torch.no_grad():
        assert ops.small_takes(x, w, glu) == tile and ops.small_takes(x, w, glu, most=rows - 1) == -1
        assert ops.small_takes(x[:, 4:], w[:, 4:], glu) == -1 and ops.small_takes(x.float(), w.float(), glu) == -1


def test_rows_far_apart():
    """what the copies' 32-bit offsets do not reach is not taken (and refused by the kernel)"""
    from timeviper_amd import kernels as ops
    flat, out = torch.empty(1024 * 1_700_000 + 64, device=DEV, dtype=BF), torch.empty(17, 512, device=DEV, dtype=BF)
    x, w = flat[:17 * 64].view(17, 64), flat.as_strided((1024, 64), (1_700_000 // 8 * 8, 1))
    with torch.no_grad():
        assert ops.small_takes(x, w.contiguous(), True) == 3 and ops.small_takes(x, w, True) == -1 and ops.small_takes(x, w[:512]) == 3
        assert ops.small_takes(flat.as_strided((17, 64), (1 << 22, 1)), w[:512]) == -1 and ops.small_takes(flat.as_strided((17, 64), ((1 << 22) - 8, 1)), w[:512]) == 3
    with pytest.raises(ops.TimeViperHipError):
        ops.small_linear(x, w, torch.zeros(1024, device=DEV, dtype=BF), ops.GEMM_GLU, out=out)


@pytest.mark.parametrize("frames", [1, 3])
def test_short_clips(frames, monkeypatch):
    """a block of a short clip on small tiles, and on the library where something stands around its layers"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.vit.siglip import Block
    torch.manual_seed(frames)
    blk = Block(1152, 16, 4304).to(DEV, BF).requires_grad_(False)
    x = torch.randn(frames, 729, 1152, device=DEV, dtype=BF)
    calls, real = [], ops.small_linear
    monkeypatch.setattr(ops, "small_linear", lambda x, w, *a, **k: (calls.append(w.shape[0]), real(x, w, *a, **k))[1])
    with torch.no_grad():
        got = [blk.forward_stream(x.clone(), None)]
        assert calls == ([3456, 1152, 4352, 1152] if frames == 1 else [3456, 1152])
        hooks = [m.register_forward_hook(lambda *a: None) for m in (blk.attn.qkv, blk.mlp.fc1)]
        calls.clear()
        got.append(blk.forward_stream(x.clone(), None))
        assert 3456 not in calls and 4352 not in calls
        for h in hooks:
            h.remove()
        z = x.double()
        f = lambda m: torch.nn.functional.linear if m is None else (lambda t: F.linear(t, m.weight.double(), m.bias.double()))
        n = lambda m, t: F.layer_norm(t, (1152,), m.weight.double(), m.bias.double(), m.eps)
        q, k, v = (t.transpose(1, 2).contiguous() for t in f(blk.attn.qkv)(n(blk.norm1, z)).view(frames, 729, 3, 16, 72).unbind(2))
        a = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) * 72 ** -0.5, -1)
        z = z + f(blk.attn.proj)(torch.matmul(a, v).transpose(1, 2).reshape(frames, 729, 1152))
        z = z + f(blk.mlp.fc2)(F.gelu(f(blk.mlp.fc1)(n(blk.norm2, z))))
    for y, pend in got:
        assert ((y.double() + pend.double() - z).norm() / z.norm()) < 6e-3    # (bf16 between the operators)
