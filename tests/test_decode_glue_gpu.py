"""The launches between two decoded tokens (csrc/decode_glue.hip) against torch: all whole numbers and copied bytes alike."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# shares that end inside a work-group's, rows that are not 16-byte aligned, the smallest size taken, ties, NaN, infinities
@pytest.mark.parametrize("rows,n,pad", [(1, 8192, 0), (3, 8195, 0), (2, 131072, 0), (5, 10001, 3), (33, 8260, 4), (2, 100, 0)])
@pytest.mark.parametrize("kind", ["random", "ties", "nan", "inf", "lowest"])
def test_argmax(rows, n, pad, kind):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(n + rows)
    x = torch.randn(rows, n + pad, generator=g, device=DEV)[:, :n]
    if kind == "ties":
        x = x.bfloat16().float()
        x[:, n // 3] = x[:, n - 1] = 9.0
    elif kind == "nan":
        x[:, n // 2] = x[:, n - 2] = float("nan")
        x[:, 1] = float("inf")
    elif kind == "inf":
        x.fill_(float("-inf"))
    elif kind == "lowest":
        x.fill_(torch.finfo(torch.float32).min)
        x[:, n - 1] = -1e30
    want = torch.stack([torch.where(r.isnan(), float("inf"), r).cpu().argmax() if not r.isnan().any() else r.isnan().int().cpu().argmax() for r in x])
    got = ops.argmax_rows(x)
    assert got.dtype == torch.int64 and torch.equal(got.cpu(), want)


@pytest.mark.parametrize("rows,n", [(1, 8192), (12, 32768), (2, 100)])
@pytest.mark.parametrize("lens", [0, 5, 70])
def test_counters_without_a_position(rows, n, lens):
    from timeviper_amd import kernels as ops
    x = torch.randn(rows, n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV)
    c = torch.arange(lens, dtype=torch.int32, device=DEV)
    assert torch.equal(ops.argmax_rows(x, (None, c)), x.argmax(-1)) and c.tolist() == list(range(1, lens + 1))


@pytest.mark.parametrize("B,H,D,sliced", [(1, 8, 128, True), (5, 2, 72, False), (12, 8, 128, True), (3, 1, 4, False)])
def test_append_and_count(B, H, D, sliced):
    from timeviper_amd import kernels as ops
    cap = 37
    qkv = torch.randn(B, 1, 4 * H * D, device=DEV).bfloat16()
    k, v = (qkv[..., i * H * D:(i + 1) * H * D].view(B, 1, H, D) for i in (1, 2)) if sliced else torch.randn(2, B, 1, H, D, device=DEV).bfloat16()
    kc, vc = torch.randn(2, B, cap, H, D, device=DEV).bfloat16()
    pos, lens = torch.tensor([cap - 2], device=DEV), torch.full((B,), cap - 1, dtype=torch.int32, device=DEV)
    wk, wv = kc.clone(), vc.clone()
    for _ in range(2):
        wk.index_copy_(1, pos, k)
        wv.index_copy_(1, pos, v)
        ops.kv_append(k, v, kc, vc, pos)
        ops.count_up(pos, lens)
        k, v = k * 2, v * 2
    assert torch.equal(kc, wk) and torch.equal(vc, wv) and pos.item() == cap and lens.tolist() == [cap + 1] * B
    if (H * D) % 8 == 0:                                       # full: nothing is written
        ops.kv_append(k, v, kc, vc, pos)
        assert torch.equal(kc, wk) and torch.equal(vc, wv)


def test_replayed():
    """captured once, replayed with eager work between: every replay as eager torch"""
    from timeviper_amd import kernels as ops
    x = torch.randn(4, 20000, device=DEV)
    pos, lens = torch.zeros(1, dtype=torch.int64, device=DEV), torch.ones(4, dtype=torch.int32, device=DEV)
    ops.argmax_rows(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        best = ops.argmax_rows(x)
        ops.count_up(pos, lens)
    for i in range(4):
        x.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(best.cpu(), x.cpu().argmax(-1)) and pos.item() == i + 1 and lens.tolist() == [i + 2] * 4
