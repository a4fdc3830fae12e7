"""Norms over every number of vectors a thread and with odd rests, on either side of the size from which a call streams past the caches; odd row counts where a wave
takes two rows."""
import pytest
import torch

from timeviper_amd import kernels as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}      # half the spacing of numbers just above a power of two
LINE = 144 << 20


def r(*s, dtype=torch.bfloat16, seed=0):
    return torch.randn(s, generator=torch.Generator(device=DEV).manual_seed(seed + sum(s)), device=DEV).to(dtype)


def close(got, want, extra=0.0):
    # the result's rounding, beside that of its factors in fp32: the mean square (D additions over 64 lanes and more, a relative 2^-20 is left of them), root, weight
    # (below 2^-14 fp16's numbers are 2^-24 apart)
    u, tiny = U[got.dtype], 2.0 ** -25 if got.dtype == torch.float16 else 1e-38
    assert ((got.double() - want).abs() <= (u * 1.01 + 2.0 ** -19) * want.abs() + extra + tiny).all()


def widths(dtype, threads):
    v = 4 if dtype == torch.float32 else 8
    return [v, v * (threads - 1), v * threads, v * (threads + 1), v * (2 * threads + 3), v * (3 * threads + 1), v * 4 * threads]


@pytest.mark.parametrize("dtype", list(U))
@pytest.mark.parametrize("rows", [1, 3, 0])                              # 0: just past the line
def test_rms(dtype, rows):
    for D in widths(dtype, 256)[:: 1 if rows else 3]:
        n = rows or LINE // (4 * D * dtype.itemsize) + 1
        x, d, w = r(n, D, dtype=dtype), r(n, D, dtype=dtype, seed=1), r(D, dtype=torch.float32 if D % 3 else dtype)
        norm = lambda s: s.double() * torch.rsqrt(s.double().square().mean(-1, keepdim=True) + 1e-5) * w.double()
        close(ops.rms_norm(x, w, 1e-5), norm(x))
        y, s = ops.rms_norm(x, w, 1e-5, residual=d, return_sum=True)
        assert torch.equal(s, (x.float() + d.float()).to(dtype))
        close(y, norm(s))


@pytest.mark.parametrize("dtype", list(U))
@pytest.mark.parametrize("rows", [1, 3, 0, -1])                          # 0, -1: just past the line, an even and an odd number of rows
def test_gated(dtype, rows):
    for group in widths(dtype, 64)[:: 1 if rows > 0 else 3]:
        D = 5 * group
        n = rows if rows > 0 else (LINE // (3 * D * dtype.itemsize) + 2) // 2 * 2 - rows
        wide, x, w = r(n, 2 * D, dtype=dtype), r(n, D, dtype=dtype, seed=1), r(D, dtype=dtype if group % 3 else torch.float32)
        for z in (wide[:, D:], None):
            y = ops.rmsnorm_fn(x[None], w, None, None if z is None else z[None], 1e-5, group, norm_before_gate=False)[0]
            for part in torch.arange(n, device=DEV).split(1 << 14) if n > 3 else [torch.arange(n, device=DEV)]:
                v = x[part].double() * (1 if z is None else torch.nn.functional.silu(z[part].double()))
                v = v.unflatten(1, (5, group))
                want = (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5)).flatten(1) * w.double()
                close(y[part], want, 2.0 ** -21 * float(want.abs().max()))       # (the gate: exp and reciprocal of the hardware, 2^-22 each)


@pytest.mark.parametrize("dtype", list(U))
@pytest.mark.parametrize("rows", [1, 5, 4097, 32771])                    # parameters late with a residual; eight rows a wave
def test_layer(dtype, rows):
    for D in widths(dtype, 64)[:: 1 if rows < 6 else 2]:
        x, d, w, b, rb = r(rows, D, dtype=dtype), r(rows, D, dtype=dtype, seed=1), r(D, dtype=dtype), r(D, dtype=dtype, seed=2), r(D, dtype=torch.float32, seed=3)

        def check(y, s):
            s = s.double()
            c = s - s.mean(-1, keepdim=True)
            n = c * torch.rsqrt(c.square().mean(-1, keepdim=True) + 1e-6) * w.double()
            # s - mean is off by 2^-24 of its largest terms, and so is n through the root of the variance; the sum with b by its own rounding
            off = 2.0 ** -21 * float((s.abs().amax(-1, keepdim=True) * torch.rsqrt(c.square().mean(-1, keepdim=True) + 1e-6)).max() * w.double().abs().max())
            close(y, n + b.double(), off + 2.0 ** -24 * float(n.abs().max()))
        check(ops.layer_norm(x, w, b, 1e-6), x)
        check(ops.layer_norm(x, w, b, 1e-6, row_bias=rb), x.float() + rb)
        y, s = ops.layer_norm(x, w, b, 1e-6, residual=d, return_sum=True)
        assert torch.equal(s, (x.float() + d.float()).to(dtype))
        check(y, s)


@pytest.mark.parametrize("dtype,D,past", [(torch.bfloat16, 1152, 0), (torch.bfloat16, 1152, 1), (torch.float32, 520, 3), (torch.float16, 2048, 7)])
def test_layer_on_either_side_of_the_size_that_is_stored_past_the_caches(dtype, D, past):
    """the last row count in front of the line (0), and behind it: the same bits as from calls of fewer rows"""
    rows = ((320 << 20) - 1) // (D * dtype.itemsize) + past
    x, w, b, rb = r(rows, D, dtype=dtype), r(D, dtype=dtype), r(D, dtype=dtype, seed=1), r(D, dtype=torch.float32, seed=2)
    y = ops.layer_norm(x, w, b, 1e-6, row_bias=rb)
    for part in torch.arange(rows, device=DEV).split(40000):
        assert torch.equal(y[part], ops.layer_norm(x[part], w, b, 1e-6, row_bias=rb))
