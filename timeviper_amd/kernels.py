"""Operator API of the TimeViper hot path, bound to the gfx950 kernels.

Each function keeps the NAME and ARGUMENT MEANING of the third-party operator
the reference calls (the boundary to the wheels it does not ship), so `NemotronHMamba2Mixer`
and friends read like the reference's:

    causal_conv1d_fn / causal_conv1d_update      modeling_nano.py:619-624 / :495-501
    mamba_chunk_scan_combined                    modeling_nano.py:639-653
    selective_state_update                       modeling_nano.py:528-539
    rmsnorm_fn                                   modeling_nano.py:372-380
    flash_attn_func / _flash_attention_forward   modeling_nano.py:1198-1209
    flash_attn_varlen_qkvpacked_func             flash_attention_class.py:59-66
    scaled_dot_product_attention                 cross_attention.py:310-317

torch is plumbing only (device memory, current stream).  There is no CPU or
eager fallback: tensors must live on the GPU and the HIP library must be built.
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
from typing import Optional

import torch

from . import _capi
from ._capi import TV_BF16, TV_F16, TV_F32, TimeViperHipError, check
from ._native import ops as _n

_DT = {torch.float32: TV_F32, torch.bfloat16: TV_BF16, torch.float16: TV_F16}


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise TimeViperHipError(f"unsupported dtype {t.dtype}") from None


def _gpu(*ts: Optional[torch.Tensor]) -> None:
    cur = -1
    for t in ts:
        if t is None or (cur >= 0 and t.get_device() == cur):
            continue
        if not t.is_cuda:
            raise TimeViperHipError(
                "timeviper_amd kernels run on the GPU only (got a CPU tensor); "
                "there is no CPU fallback in the product path"
            )
        # the launch goes to the CURRENT device's stream (`_stream`): a tensor of another device
        # would hand that stream foreign pointers.  One process drives one GPU here.
        # (a GPU tensor exists: torch.cuda.current_device()'s look at the initialisation is half of its time)
        cur = torch._C._cuda_getDevice()
        if t.get_device() != cur:
            raise TimeViperHipError(
                f"tensor on cuda:{t.get_device()} but the current device is cuda:{cur}: "
                "call torch.cuda.set_device() (one process per GPU)")


def _stream() -> int:
    # the handle alone: a torch.cuda.Stream object around it takes 6 us of every launch
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _p(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _as(t: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """t, dense and of `dtype` (two calls into torch saved where it is both)"""
    return t if t.dtype is dtype and t.is_contiguous() else t.to(dtype).contiguous()


def _like_rows(t: torch.Tensor):
    """(rows, row stride, empty tensor of t's shape) of dense t, without the views that `_rows2d` makes; else None"""
    D = t.shape[-1]
    if D == 0 or not t.is_contiguous():
        return None
    return t.numel() // D, D, torch.empty_like(t, memory_format=torch.contiguous_format)


def _rows2d(t: torch.Tensor) -> torch.Tensor:
    """View (..., D) as (rows, D) with one row stride, copying only if needed."""
    if t.stride(-1) != 1:
        t = t.contiguous()
    if t.dim() == 2:
        return t
    try:
        return t.view(-1, t.shape[-1])
    except RuntimeError:
        return t.reshape(-1, t.shape[-1])


# --------------------------------------------------------------------- conv1d
def causal_conv1d_fn(x, weight, bias=None, seq_idx=None, initial_states=None,
                     return_final_states=False, final_states_out=None, activation=None,
                     halo=None):
    """x: (B, C, L) — the reference passes the transposed view of a (B, L, C)
    tensor, which is exactly the channels-last layout the kernel wants.
    weight (C, K), bias (C).  Returns (B, C, L) (again a transposed view).
    `halo` (B, K-1, C): rows preceding this shard (sequence sharding)."""
    if seq_idx is not None or initial_states is not None or return_final_states:
        raise TimeViperHipError("causal_conv1d_fn: seq_idx/initial_states/final_states unsupported")
    if activation not in (None, "silu", "swish"):
        raise TimeViperHipError(f"causal_conv1d_fn: activation {activation!r}")
    _gpu(x, weight, bias, halo)
    B, Cc, L = x.shape
    xl = x.transpose(1, 2)  # (B, L, C)
    if xl.stride(2) != 1:
        xl = xl.contiguous()
    K = weight.shape[-1]
    w = weight.reshape(Cc, K).to(x.dtype).contiguous()
    b = None if bias is None else bias.to(x.dtype).contiguous()
    if halo is not None:
        halo = halo.to(x.dtype).contiguous()
        assert halo.shape == (B, K - 1, Cc)
    y = torch.empty((B, L, Cc), dtype=x.dtype, device=x.device)
    check(_capi.lib().tv_causal_conv1d_fwd(
        _p(xl), _p(w), _p(b), _p(halo), _p(y), B, L, Cc, K, xl.stride(0), xl.stride(1),
        y.stride(0), y.stride(1), _dt(x), int(activation in ("silu", "swish")), _stream()),
        "tv_causal_conv1d_fwd")
    return y.transpose(1, 2)


def causal_conv1d_xbc(xBC, weight, bias, d_inner: int, ngroups: int, dstate: int,
                      activation="silu", halo=None, return_cb: bool = False):
    """Mamba-2 mixer variant of causal_conv1d_fn + the [x | B | C] split of
    modeling_nano.py:628-636 in one pass.  xBC (B, L, d_inner + 2*G*N) (any row stride).
    Returns x (B, L, d_inner) and B, C as (B, L, G, N) VIEWS of group-major (B, G, L, N)
    storage — the layout the scan kernel streams best.
    `return_cb`: also return the causal C.B^T fragments of every (chunk, group) for
    `mamba_chunk_scan_combined(..., cb=...)` (an opaque bf16 tensor; None where the scan would
    not use them: other dtypes / d_state), computed while the B / C tiles are on the chip."""
    if halo is None and xBC.is_cuda and (r := _n.conv_xbc(xBC, weight, bias, d_inner, ngroups, dstate, activation in ("silu", "swish"), return_cb)) is not None:
        return r
    _gpu(xBC, weight, bias, halo)
    Bsz, L, Cc = xBC.shape
    assert Cc == d_inner + 2 * ngroups * dstate
    if xBC.stride(2) != 1:
        xBC = xBC.contiguous()
    K = weight.shape[-1]
    w = _as(weight if weight.dim() == 2 else weight.reshape(Cc, K), xBC.dtype)
    if w.shape[0] != Cc:
        w = w.reshape(Cc, K)
    b = None if bias is None else _as(bias, xBC.dtype)
    if halo is not None:
        halo = _as(halo, xBC.dtype)
    yx = xBC.new_empty((Bsz, L, d_inner))
    yb = xBC.new_empty((Bsz, ngroups, L, dstate))
    yc = torch.empty_like(yb)
    lib = _capi.lib()
    if return_cb and xBC.dtype == torch.bfloat16 and dstate == 128 and L > 0:
        cb = torch.empty(lib.tv_ssd_cb_bytes(Bsz, L, ngroups) // 2, dtype=torch.bfloat16, device=xBC.device)
        check(lib.tv_causal_conv1d_xbc_cb_fwd(
            _p(xBC), _p(w), _p(b), _p(halo), _p(yx), _p(yb), _p(yc), _p(cb), Bsz, L, d_inner, ngroups, dstate,
            K, xBC.stride(0), xBC.stride(1), _dt(xBC), int(activation in ("silu", "swish")), _stream()),
            "tv_causal_conv1d_xbc_cb_fwd")
        return yx, yb.transpose(1, 2), yc.transpose(1, 2), cb
    check(lib.tv_causal_conv1d_xbc_fwd(
        _p(xBC), _p(w), _p(b), _p(halo), _p(yx), _p(yb), _p(yc), Bsz, L, d_inner, ngroups, dstate,
        K, xBC.stride(0), xBC.stride(1), _dt(xBC), int(activation in ("silu", "swish")), _stream()),
        "tv_causal_conv1d_xbc_fwd")
    if return_cb:
        return yx, yb.transpose(1, 2), yc.transpose(1, 2), None
    return yx, yb.transpose(1, 2), yc.transpose(1, 2)


def causal_conv1d_update(x, conv_state, weight, bias=None, activation=None):
    """x (B, C); conv_state (B, C, K) updated in place; returns (B, C)."""
    _gpu(x, conv_state, weight, bias)
    B, Cc = x.shape
    K = weight.shape[-1]
    if not conv_state.is_contiguous() or conv_state.dtype != x.dtype:
        raise TimeViperHipError("causal_conv1d_update: conv_state must be contiguous, x.dtype")
    xc = x.contiguous()
    w = weight.reshape(Cc, K).to(x.dtype).contiguous()
    b = None if bias is None else bias.to(x.dtype).contiguous()
    y = torch.empty_like(xc)
    check(_capi.lib().tv_causal_conv1d_update(
        _p(xc), _p(conv_state), _p(w), _p(b), _p(y), B, Cc, K, _dt(x),
        int(activation in ("silu", "swish")), _stream()), "tv_causal_conv1d_update")
    return y


# ---------------------------------------------------------------------- norms
def rms_norm(x, weight, eps, residual=None, return_sum=False):
    """NemotronHRMSNorm (modeling_nano.py:897-903); with `residual`, normalises
    s = x + residual (rounded to x.dtype like the reference's bf16 add, :966) and
    can return s too."""
    if x.is_cuda and (r := _n.rms_norm(x, weight, eps, residual, return_sum)) is not None:
        return r
    _gpu(x, weight, residual)
    w = weight if weight.dtype in (torch.float32, x.dtype) else weight.to(torch.float32)
    w = w.contiguous()
    dense = _like_rows(x) if residual is None or (residual.is_contiguous() and residual.shape == x.shape) else None
    if dense:
        (n, D, y), s = dense, torch.empty_like(x) if return_sum and residual is not None else None
        check(_capi.lib().tv_rmsnorm_fwd(_p(x), _p(residual), _p(w), _p(s), _p(y), n, D, D, 0 if residual is None else D, 0 if s is None else D, D, float(eps),
                                         _dt(x), _dt(w), _stream()), "tv_rmsnorm_fwd")
        return (y, x if s is None else s) if return_sum else y
    x2 = _rows2d(x)
    r2 = None if residual is None else _rows2d(residual)
    y = torch.empty(x2.shape, dtype=x.dtype, device=x.device)
    s = torch.empty_like(y) if (return_sum and residual is not None) else None
    check(_capi.lib().tv_rmsnorm_fwd(
        _p(x2), _p(r2), _p(w), _p(s), _p(y), x2.shape[0], x2.shape[1], x2.stride(0),
        0 if r2 is None else r2.stride(0), 0 if s is None else s.stride(0), y.stride(0),
        float(eps), _dt(x), _dt(w), _stream()), "tv_rmsnorm_fwd")
    y = y.view(x.shape)
    if return_sum:
        return y, (s.view(x.shape) if s is not None else x)
    return y


def layer_norm(x, weight, bias, eps, residual=None, return_sum=False, row_bias=None):
    """nn.LayerNorm over the last dim, optionally of s = x + residual (rounded to x.dtype),
    returning s too — the fused form of a pre-norm ViT block's residual add + norm.
    `row_bias` (D,) fp32: a constant row added to every s before the statistics (not to the
    returned sum): the projection biases a caller carries beside a stream its GEMMs accumulate into."""
    if residual is None and x.is_cuda and (r := _n.layer_norm(x, weight, bias, eps, return_sum, row_bias)) is not None:
        return r
    _gpu(x, weight, bias, residual, row_bias)
    w = _as(weight, x.dtype)
    b = None if bias is None else _as(bias, x.dtype)
    rb = None if row_bias is None else _as(row_bias, torch.float32)
    dense = _like_rows(x) if residual is None else None
    if dense:
        n, D, y = dense
        check(_capi.lib().tv_layernorm_fwd(_p(x), None, _p(w), _p(b), _p(rb), None, _p(y), n, D, D, 0, 0, D, float(eps), _dt(x), _stream()), "tv_layernorm_fwd")
        return (y, x) if return_sum else y
    x2 = _rows2d(x)
    r2 = None if residual is None else _rows2d(residual)
    y = torch.empty(x2.shape, dtype=x.dtype, device=x.device)
    s = torch.empty_like(y) if (return_sum and residual is not None) else None
    check(_capi.lib().tv_layernorm_fwd(
        _p(x2), _p(r2), _p(w), _p(b), _p(rb), _p(s), _p(y), x2.shape[0], x2.shape[1], x2.stride(0),
        0 if r2 is None else r2.stride(0), 0 if s is None else s.stride(0), y.stride(0), float(eps),
        _dt(x), _stream()), "tv_layernorm_fwd")
    y = y.view(x.shape)
    if return_sum:
        return y, (s.view(x.shape) if s is not None else x)
    return y


def gelu(x, inplace=False):
    """exact (erf) GELU, elementwise."""
    _gpu(x)
    xc = x if x.is_contiguous() else x.contiguous()
    y = xc if inplace else torch.empty_like(xc)
    check(_capi.lib().tv_gelu_fwd(_p(xc), _p(y), xc.numel(), _dt(xc), _stream()), "tv_gelu_fwd")
    return y


def relu2(x, inplace=False):
    """square(relu(x)) — NemotronHMLP's activation (modeling_nano.py:993-994), elementwise."""
    _gpu(x)
    xc = x if x.is_contiguous() else x.contiguous()
    y = xc if inplace else torch.empty_like(xc)
    check(_capi.lib().tv_relu2_fwd(_p(xc), _p(y), xc.numel(), _dt(xc), _stream()), "tv_relu2_fwd")
    return y


def rmsnorm_fn(x, weight, bias=None, z=None, eps=1e-6, group_size=None,
               norm_before_gate=True, upcast=True):
    """mamba_ssm.ops.triton.layernorm_gated.rmsnorm_fn as the reference calls it
    (norm_before_gate=False): y = w * u * rsqrt(mean_group(u^2)+eps), u = x*silu(z)."""
    if bias is not None:
        raise TimeViperHipError("rmsnorm_fn: bias unsupported (reference passes None)")
    if z is not None and norm_before_gate:
        raise TimeViperHipError("rmsnorm_fn: only norm_before_gate=False is on the path")
    if x.is_cuda and (r := _n.gated_norm(x, weight, z, eps, group_size)) is not None:
        return r
    _gpu(x, weight, z)
    D = x.shape[-1]
    gs = D if group_size is None else int(group_size)
    w = weight if weight.dtype in (torch.float32, x.dtype) else weight.to(torch.float32)
    w = w.contiguous()
    # (z: a slice of a wider projection, whose rows of one batch entry lie one distance apart)
    if z is None or (z.dim() == 3 and z.shape == x.shape and z.stride(2) == 1 and (z.shape[0] == 1 or z.stride(0) == z.shape[1] * z.stride(1))):
        dense = _like_rows(x)
        if dense:
            n, _, y = dense
            check(_capi.lib().tv_rmsnorm_gated_fwd(_p(x), _p(z), _p(w), _p(y), n, D, gs, D, 0 if z is None else z.stride(1), D, float(eps), _dt(x), _dt(w),
                                                   _stream()), "tv_rmsnorm_gated_fwd")
            return y
    x2 = _rows2d(x)
    z2 = None if z is None else _rows2d(z)
    y = torch.empty(x2.shape, dtype=x.dtype, device=x.device)
    check(_capi.lib().tv_rmsnorm_gated_fwd(
        _p(x2), _p(z2), _p(w), _p(y), x2.shape[0], D, gs, x2.stride(0),
        0 if z2 is None else z2.stride(0), y.stride(0), float(eps), _dt(x), _dt(w), _stream()),
        "tv_rmsnorm_gated_fwd")
    return y.view(x.shape)


# ------------------------------------------------------------------- linears with fused epilogues
CUS = 256            # compute units of an MI355X: work-groups of one round
GEMM_BIAS, GEMM_BIAS_GELU, GEMM_ACCUM, GEMM_BIAS_RELU2 = 0, 1, 2, 3


def linear_fused(x, weight, bias=None, epilogue: int = GEMM_BIAS, out=None):
    """F.linear(x, weight, bias) on the hand-written bf16 GEMM (csrc/gemm.hip) with the epilogue fused:
    GEMM_BIAS (plain), GEMM_BIAS_GELU (exact GELU of the bf16-rounded result: the timm Mlp's fc1 + act), GEMM_BIAS_RELU2 (its squared
    ReLU; at least 256 rows and columns, on the persistent kernel alone) or GEMM_ACCUM (out += x @ weight.T, `out` required, bias ignored).  x (..., K) bf16 with dense rows,
    weight (N, K) bf16; K % 128 == 0, N % 4 == 0."""
    _gpu(x, weight, bias, out)
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TimeViperHipError("linear_fused: bf16 only")
    x2 = _rows2d(x)
    N, Kd = weight.shape
    if weight.stride(1) != 1:
        weight = weight.contiguous()
    if out is None and epilogue in (GEMM_BIAS, GEMM_BIAS_RELU2) and Kd >= 4096 and Kd % 128 == 0 and x.shape[-1] == Kd and x2.stride(0) % 8 == 0 \
            and weight.stride(0) % 8 == 0 and (x2.data_ptr() | weight.data_ptr()) % 16 == 0 and bias is None and N % 8 == 0 and gemm_persist_on():
        plan = tail_plan(x2.shape[0], N, Kd)
        if plan:
            return split_linear(x2.view(x.shape), weight, None, epilogue == GEMM_BIAS_RELU2, *plan)
    if epilogue == GEMM_ACCUM:
        if out is None:
            raise TimeViperHipError("linear_fused: GEMM_ACCUM needs `out`")
        bias = None
    if out is None:
        out = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    o2 = out.view(-1, N) if out.dim() != 2 else out
    if o2.stride(1) != 1 or o2.shape[0] != x2.shape[0]:
        raise TimeViperHipError("linear_fused: `out` must be (rows, N) with a contiguous last dim")
    bd = TV_F32
    if bias is not None:
        if bias.dtype not in (torch.float32, torch.bfloat16):
            bias = bias.float()
        bias = bias.contiguous()
        bd = _dt(bias)
    lib, rows = _capi.lib(), x2.shape[0]
    lead = lead_rows(rows, N, Kd, epilogue)
    if lead and ((x2.data_ptr() | weight.data_ptr() | o2.data_ptr() | (0 if bias is None else bias.data_ptr())) % 16 or x2.stride(1) != 1
                 or (x2.stride(0) | weight.stride(0) | o2.stride(0)) % 8 or x2.shape[1] != Kd or max(x2.stride(0), weight.stride(0)) >= (1 << 22)
                 or (bias is not None and bd == TV_F32) or not gemm_persist_on()):         # (an fp32 bias may take launches of many tiles to another kernel)
        lead = 0
    check(lib.tv_gemm_bf16_fwd(_p(x2), _p(weight), _p(bias), _p(o2), lead or rows, N, Kd, x2.stride(0), weight.stride(0), o2.stride(0), int(epilogue), bd, _stream()),
          "tv_gemm_bf16_fwd")
    if lead:
        check(lib.tv_gemm_small_fwd(_p(x2[lead:]), _p(weight), _p(bias), _p(o2[lead:]), rows - lead, N, Kd, x2.stride(0), weight.stride(0), o2.stride(0),
                                    int(epilogue), bd, 0, _stream()), "tv_gemm_small_fwd")
    return out


def lead_rows(rows: int, n: int, k: int, epilogue: int) -> int:
    """The rows in front of a product of short contraction that fill whole rounds of 256 x 256 tiles, where the rows behind them are one 128 x 128 tile a compute
    unit or less: such a launch (csrc/gemm_small.hip) takes 15 us where a round that is nearly empty takes a full one's 26 - 35; 0: all rows in one launch.
    us, one launch | two, n x k 4 352 x 1 152 with the GELU: 4 374 rows, 1.2 rounds, 67 | 56, 8 180: 108 | 94, 12 320: 143 | 132, 20 000, 5.3: 221 | 207, 35 060:
    364 | 359; 4 096 x 1 024: 4 896: 63 | 54; 3 072 x 768: 11 552: 85 | 77; 8 192 x 2 048: 2 548: 99 | 85, 10 740: 311 | 302; plain, up to three rounds, 3 456 x 1 152:
    5 103: 52 | 47, 10 016: 86 | 81, 23 552: 168 | 173; 6 144 x 2 048: 3 060: 84 | 75.  With 270 small tiles and more (10 416 rows: 85 | 87) the second
    round of them costs what it saves."""
    if epilogue not in (GEMM_BIAS, GEMM_BIAS_GELU) or not 768 <= k <= 2048 or n < 2048 or n % 8 or k % 128:
        return 0
    wide = -(-n // 256)
    rounds = -(-rows // 256) * wide // CUS
    lead = rounds * CUS // wide * 256
    if rounds < 1 or lead >= rows or (epilogue == GEMM_BIAS and rounds > 3) or -(-(rows - lead) // 128) * -(-n // 128) > CUS:
        return 0
    return lead


def param_key(params):
    """Cache key for tensors derived from parameters (stacked / padded / fp32 copies): storage, version counter, dtype
    and device of each.  Tensors created under `torch.inference_mode()` track no version ("Inference tensors do not
    track version counter"): they count as version 0 — such a model must not be written in place after its first forward.
    Note that writes through `.data` never bump the counter either: reload weights with `load_state_dict` / `copy_`."""
    # (asked first: the exception that `_version` of an inference tensor raises takes 15 us, 2.6 ms of a four-frame clip's 7.1)
    return tuple([(p.data_ptr(), 0 if p.is_inference() else p._version, p.dtype, p.device) for p in params])


def gemm_set_persist(mode: int = -1, grid: int = 0) -> None:
    """Which of the two GEMM kernels `linear_fused` runs on: -1 automatic and 1 the persistent kernel
    wherever the shape allows, 0 the per-tile kernel only; `grid`:
    work-groups of the persistent kernel (0 = one per compute unit; tests use 8 so that small problems still give
    every work-group several tiles)."""
    _capi.lib().tv_gemm_set_persist(int(mode), int(grid))


def gemm_persist_on() -> bool:
    """Whether `linear_fused` may take the persistent kernel (`gemm_set_persist`, TV_GEMM_PERSIST)."""
    return bool(_capi.lib().tv_gemm_persist_on())


# zero-padded inference copies of weights (model/vit/siglip.py): storage address -> (useful rows, useful columns), so that a
# FLOP count (bench.py) can leave the padding out whatever view of the copy a GEMM receives
PADDED_USEFUL: dict = {}


def gemm_set_drip(mode: int = -1) -> None:
    """The 256 x 192-tile persistent GEMM (csrc/gemm_drip.hip): -1 automatic (first choice wherever the shape allows and
    every compute unit gets a few tiles), 0 never, 1 wherever the shape allows (tests on small grids)."""
    _capi.lib().tv_gemm_set_drip(int(mode))


# ------------------------------------------------------------------- SSD scan
def _row_view(t: torch.Tensor, inner: int):
    """(B, L, ...) tensor whose trailing dims are contiguous with `inner`
    elements per row: return (tensor, stride_b, stride_l) without copying when
    the rows are dense (slices of a wider projection keep their row stride)."""
    if t.is_contiguous():
        return t, t.stride(0), t.stride(1)
    ok = t.stride(-1) == 1
    exp = 1
    for d in range(t.dim() - 1, 1, -1):
        ok = ok and t.stride(d) == exp
        exp *= t.shape[d]
    if not ok:
        t = t.contiguous()
    return t, t.stride(0), t.stride(1)


def mamba_chunk_scan_combined(x, dt, A, B, C, chunk_size=None, D=None, z=None, dt_bias=None,
                              initial_states=None, seq_idx=None, cu_seqlens=None,
                              dt_softplus=False, dt_limit=(0.0, float("inf")),
                              return_final_states=False, return_varlen_states=False,
                              group_map="block", return_total_decay=False, cb=None):
    """x (B,L,H,P), dt (B,L,H), A (H), B/C (B,L,G,N), D (H), dt_bias (H),
    initial_states (B,H,P,N).  Returns y (B,L,H,P) [, final_states (B,H,P,N) fp32]
    [, total_decay (B,H) fp32].  `chunk_size` is accepted for signature parity
    and ignored (the result is chunk-invariant).  `group_map`: "block"
    (h // (H/G), GPU reference) or "tile" (h % G, reference CPU quirk).
    `cb`: the C.B^T fragments `causal_conv1d_xbc(..., return_cb=True)` returned for these B / C."""
    if z is not None or seq_idx is not None or cu_seqlens is not None or return_varlen_states:
        raise TimeViperHipError("mamba_chunk_scan_combined: z/seq_idx/cu_seqlens unsupported")
    if D is not None and D.dim() != 1:
        raise TimeViperHipError("mamba_chunk_scan_combined: D must be (nheads,)")
    if x.is_cuda and (r := _n.scan(x, dt, A, B, C, D, dt_bias, initial_states, dt_softplus, dt_limit[0], min(dt_limit[1], 3.0e38), return_final_states, return_total_decay,
                                   {"block": 0, "tile": 1}[group_map], cb)) is not None:
        return r
    _gpu(x, dt, A, B, C, D, dt_bias, initial_states)
    Bsz, L, H, P = x.shape
    G, N = B.shape[2], B.shape[3]
    if dt.dtype != x.dtype:
        dt = dt.to(x.dtype)
    if B.dtype != x.dtype:
        B = B.to(x.dtype)
    if C.dtype != x.dtype:
        C = C.to(x.dtype)
    x, xsb, xsl = _row_view(x, H * P)
    dt, dsb, dsl = _row_view(dt, H)
    # B/C: any (B, L, G, N) view with contiguous N (token-major rows or group-major storage)
    if B.stride(3) != 1:
        B = B.contiguous()
    if C.stride(3) != 1:
        C = C.contiguous()
    bsb, bsl, bsg = B.stride(0), B.stride(1), B.stride(2)
    csb, csl, csg = C.stride(0), C.stride(1), C.stride(2)
    f32 = lambda t: None if t is None else _as(t, torch.float32)
    A, D, dt_bias, initial_states = f32(A), f32(D), f32(dt_bias), f32(initial_states)
    y = x.new_empty((Bsz, L, H, P))
    final = torch.empty((Bsz, H, P, N), dtype=torch.float32, device=x.device) \
        if return_final_states else None
    decay = torch.empty((Bsz, H), dtype=torch.float32, device=x.device) \
        if return_total_decay else None
    lib = _capi.lib()
    ws_bytes = lib.tv_ssd_scan_workspace_bytes(Bsz, L, H, P, G, N, _dt(x))
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=x.device)
    if cb is not None:
        _gpu(cb)
        if cb.dtype != torch.bfloat16 or cb.numel() * 2 != lib.tv_ssd_cb_bytes(Bsz, L, G) or not cb.is_contiguous():
            raise TimeViperHipError("mamba_chunk_scan_combined: cb is not the C.B^T buffer of these shapes")
    check(lib.tv_ssd_scan_cb_fwd(
        _p(x), _p(dt), _p(A), _p(B), _p(C), _p(cb), _p(D), _p(dt_bias), _p(initial_states), _p(y),
        _p(final), _p(decay), Bsz, L, H, P, G, N, xsb, xsl, dsb, dsl, bsb, bsl, bsg, csb, csl, csg,
        y.stride(0), y.stride(1), _dt(x), int(bool(dt_softplus)), float(dt_limit[0]),
        float(min(dt_limit[1], 3.0e38)), {"block": 0, "tile": 1}[group_map], _p(ws), ws_bytes,
        _stream()), "tv_ssd_scan_cb_fwd")
    out = (y,)
    if return_final_states:
        out += (final,)
    if return_total_decay:
        out += (decay,)
    return out[0] if len(out) == 1 else out


def ssd_state_correction(y, dt, A, C, state_in, dt_bias=None, dt_softplus=False,
                         dt_limit=(0.0, float("inf")), group_map="block"):
    """In place: y_t += exp(sum_{j<=t} dt_j A_h) C_t . state_in[h] — completes the outputs of a scan
    that started from a zero state once the state entering it is known (sequence
    shards).  y (B,L,H,P), dt (B,L,H) raw, C (B,L,G,N), state_in (B,H,P,N) fp32.  Returns y."""
    _gpu(y, dt, A, C, state_in, dt_bias)
    Bsz, L, H, P = y.shape
    G, N = C.shape[2], C.shape[3]
    assert y.stride(3) == 1 and y.stride(2) == P, "y rows must be dense (H*P elements)"
    if dt.dtype != y.dtype:
        dt = dt.to(y.dtype)
    dt, dsb, dsl = _row_view(dt, H)
    if C.dtype != y.dtype:
        C = C.to(y.dtype)
    if C.stride(3) != 1:
        C = C.contiguous()
    f32 = lambda t: None if t is None else t.to(torch.float32).contiguous()
    A, dt_bias, state_in = f32(A), f32(dt_bias), f32(state_in)
    lib = _capi.lib()
    ws_bytes = lib.tv_ssd_state_correction_workspace_bytes(Bsz, L, H)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=y.device)
    check(lib.tv_ssd_state_correction(
        _p(y), _p(dt), _p(A), _p(C), _p(dt_bias), _p(state_in), Bsz, L, H, P, G, N,
        y.stride(0), y.stride(1), dsb, dsl, C.stride(0), C.stride(1), C.stride(2), _dt(y),
        int(bool(dt_softplus)), float(dt_limit[0]), float(min(dt_limit[1], 3.0e38)),
        {"block": 0, "tile": 1}[group_map], _p(ws), ws_bytes, _stream()), "tv_ssd_state_correction")
    return y


def selective_state_update(state, x, dt, A, B, C, D=None, z=None, dt_bias=None,
                           dt_softplus=False):
    """Single decode step.  state (B,H,P,N) fp32, in place.  The reference passes
    A/dt/dt_bias/D expanded over (P[,N]) from per-head values (:514-522); the
    kernel takes the per-head values, so expanded views are reduced here."""
    if z is not None:
        raise TimeViperHipError("selective_state_update: z unsupported (reference passes None)")
    _gpu(state, x, dt, A, B, C, D, dt_bias)
    Bsz, H, P = x.shape
    G, N = B.shape[1], B.shape[2]
    if state.dtype != torch.float32 or not state.is_contiguous():
        raise TimeViperHipError("selective_state_update: state must be contiguous fp32")
    head = lambda t, nd: None if t is None else \
        (t if t.dim() == nd else t[(..., *([0] * (t.dim() - nd)))]).to(torch.float32).contiguous()
    A1, D1, b1 = head(A, 1), head(D, 1), head(dt_bias, 1)
    # slices of the mixer's projection are read in place (one row per sequence, dense behind the batch dimension)
    rows = lambda t: t if t.stride(1) == t.shape[2] and t.stride(2) == 1 and t.data_ptr() % 16 == 0 and t.stride(0) % 8 == 0 else t.contiguous()
    dt1 = (dt if dt.dim() == 2 else dt[..., 0]).to(x.dtype)
    dt1 = dt1 if dt1.stride(1) == 1 else dt1.contiguous()
    xc, Bc, Cc = rows(x), rows(B.to(x.dtype)), rows(C.to(x.dtype))
    y = torch.empty((Bsz, H, P), dtype=x.dtype, device=x.device)
    check(_capi.lib().tv_selective_state_update_rows(
        _p(state), _p(xc), _p(dt1), _p(A1), _p(Bc), _p(Cc), _p(D1), _p(b1), _p(y), Bsz, H, P, G,
        N, xc.stride(0), dt1.stride(0), Bc.stride(0), Cc.stride(0), _dt(x), int(bool(dt_softplus)), _stream()),
        "tv_selective_state_update_rows")
    return y


def ssd_scan_set_impl(impl: int) -> None:
    """0 auto (= 6 where it applies, else 4, 3; other dtypes / d_state: 8, else 1), 1 generic fp32 token recurrence, 3 MFMA
    slice march on <= 40-column slices of a head, 4 whole-head slice march x sequence segments, 6 head-per-wave march
    (ssd_head.hip, at every length), 8 chunk-parallel fp32 form (ssd_chunked.hip); 2 / 5 / 7 (removed kernels) select 3 / 4 / 6.
    Process-global (dev tools and tests)."""
    _capi.lib().tv_ssd_scan_set_impl(int(impl))


def ssd_head_set_asm(on: int) -> None:
    """Head-per-wave march at head_dim 80 x 4 heads per work-group: 1 the generated step (default), 0 the C++ step, -1 default /
    TV_HEAD_ASM.  Process-global (A/B runs and the bit-identity test)."""
    _capi.lib().tv_ssd_head_set_asm(int(on))


def ssd_scan_last_impl() -> int:
    """Kernel family (the numbers of `ssd_scan_set_impl`) the most recent scan call of this process ran on."""
    return int(_capi.lib().tv_ssd_scan_last_impl())


def ssd_scan_last_kernel() -> int:
    """The kernel of that call: the same numbers, and those that only automatic selection takes: 9 column slices (ssd_cols.hip) and 10 a head per work-group in
    segments (ssd_par.hip), of family 6; 11 chunks on the fp32 matrix instruction (ssd_f32.hip), of family 8."""
    return int(_capi.lib().tv_ssd_scan_last_kernel())


# ------------------------------------------------------------------ attention
def flash_attn_set_variant(variant: int) -> None:
    """0 auto (bf16 ViT frames: the kernel with the generated tile loop, csrc/attention_vit.hpp; else the compiled streaming
    kernel), 5 always the compiled streaming kernel (P's row sums out of the P.V MFMAs), 3 the compiled kernel with the row
    sums on the vector pipe (A/B, tests); include/timeviper_hip.h.  Process-global (dev tools and tests)."""
    _capi.lib().tv_flash_attn_set_variant(int(variant))


_ATTN_FP8 = {"on": False, "min_keys": 4096, "min_queries": 64}


class fp8_attention:
    """Context manager / switch: inside it `flash_attn_func` (and everything built on it) runs the
    QK^T / PV products on the FP8 MFMA path (`tv_flash_attn_fp8_fwd`).  Off by
    default: the reference's attention arithmetic is bf16.  Key sequences shorter than `min_keys`
    stay on the bf16 kernel: the ViT towers (<= 1 025 keys per frame / tube; measured 2.3 ms fp8
    against 1.5 ms bf16 per 256 SigLIP frames — the quantisation pre-pass and head_dim 72 -> 128
    padding cost more than the MFMAs save); calls with fewer than `min_queries` queries stay there too: the
    decode step (one query against the whole cache: the quantisation pre-pass over the cache would cost
    more than the attention, with per-head scales that differ from the prefill's).  The long causal LM
    attention is where the fp8 matrix rate pays (131 172 tokens, 28/4 x 128: 83 ms against 122 ms).
    The switch is process-global state (like `ssd_scan_set_impl`): right for an evaluation process, not for
    two models with different settings in one process."""

    def __init__(self, on: bool = True, min_keys: int = 4096, min_queries: int = 64):
        self.new = {"on": bool(on), "min_keys": int(min_keys), "min_queries": int(min_queries)}

    def __enter__(self):
        self.old = dict(_ATTN_FP8)
        _ATTN_FP8.update(self.new)
        return self

    def __exit__(self, *exc):
        _ATTN_FP8.update(self.old)


def flash_attn_fp8_func(q, k, v, softmax_scale=None, causal=False, return_lse=False):
    """`flash_attn_func` with e4m3 MFMA operands (per-head scales, fp32 accumulation / softmax)."""
    _gpu(q, k, v)
    B, Lq, Hq, D = q.shape
    Lk, Hkv = k.shape[1], k.shape[2]
    fix = lambda t: t if t.stride(-1) == 1 else t.contiguous()
    q, k, v = fix(q), fix(k), fix(v)
    if D % 8 or D > 128:
        raise TimeViperHipError(f"flash_attn_fp8_func: head_dim {D} must be a multiple of 8, <= 128")
    for t in (q, k, v):
        if any(s % 8 for s in t.stride()[:3]) or t.data_ptr() % 16:
            raise TimeViperHipError("flash_attn_fp8_func: strides must be multiples of 8 elements")
    scale = 1.0 / math.sqrt(D) if softmax_scale is None else float(softmax_scale)
    o = torch.empty((B, Lq, Hq, D), dtype=q.dtype, device=q.device)
    lse = torch.empty((B, Hq, Lq), dtype=torch.float32, device=q.device) if return_lse else None
    lib = _capi.lib()
    ws_bytes = lib.tv_flash_attn_fp8_workspace_bytes(B, Lq, Lk, Hq, Hkv)
    ws = torch.empty(max(ws_bytes, 256), dtype=torch.uint8, device=q.device)
    check(lib.tv_flash_attn_fp8_fwd(
        _p(q), _p(k), _p(v), _p(o), _p(lse), B, Lq, Lk, Hq, Hkv, D,
        q.stride(0), q.stride(1), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
        v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(1), o.stride(2),
        scale, int(bool(causal)), _dt(q), _p(ws), ws_bytes, _stream()), "tv_flash_attn_fp8_fwd")
    return (o, lse) if return_lse else o


def flash_attn_func(q, k, v, dropout_p=0.0, softmax_scale=None, causal=False,
                    return_lse=False):
    """q (B,Lq,Hq,D), k/v (B,Lk,Hkv,D) -> (B,Lq,Hq,D).  GQA without repeat_kv;
    causal mask bottom-right aligned (flash-attn >= 2.1 semantics)."""
    if dropout_p:
        raise TimeViperHipError("flash_attn_func: dropout is not on the inference path")
    if q.is_cuda and not _ATTN_FP8["on"] and (r := _n.flash(q, k, v, softmax_scale, causal, return_lse)) is not None:
        return r
    _gpu(q, k, v)
    B, Lq, Hq, D = q.shape
    Lk, Hkv = k.shape[1], k.shape[2]
    # (Lq >= 64: a decode step against a long cache stays on the bf16 kernel — the fp8 path would re-quantise and
    # transpose the whole K / V cache for one query, with a scale that differs from the prefill's)
    if _ATTN_FP8["on"] and Lk >= _ATTN_FP8["min_keys"] and Lq >= _ATTN_FP8["min_queries"] and D <= 128 \
            and q.dtype in (torch.bfloat16, torch.float16):
        return flash_attn_fp8_func(q, k, v, softmax_scale, causal, return_lse)
    fix = lambda t: t if t.stride(-1) == 1 else t.contiguous()
    q, k, v = fix(q), fix(k), fix(v)
    if Lq == 1 and _decode_attn_takes(q, k, v):         # a decode step: split-KV kernel (causal or not: one query, last row)
        return flash_attn_decode(q, k, v, softmax_scale=softmax_scale, return_lse=return_lse)
    if D % 8:
        raise TimeViperHipError(f"flash_attn_func: head_dim {D} must be a multiple of 8")
    strides = q.stride()[:3] + k.stride()[:3] + v.stride()[:3]
    if any([s % 8 for s in strides]) or (q.data_ptr() | k.data_ptr() | v.data_ptr()) % 16:
        raise TimeViperHipError("flash_attn_func: strides must be multiples of 8 elements")
    scale = 1.0 / math.sqrt(D) if softmax_scale is None else float(softmax_scale)
    o = torch.empty((B, Lq, Hq, D), dtype=q.dtype, device=q.device)
    lse = torch.empty((B, Hq, Lq), dtype=torch.float32, device=q.device) if return_lse else None
    check(_capi.lib().tv_flash_attn_fwd(
        _p(q), _p(k), _p(v), _p(o), _p(lse), B, Lq, Lk, Hq, Hkv, D, *strides, *o.stride()[:3],
        scale, int(bool(causal)), _dt(q), _stream()), "tv_flash_attn_fwd")
    return (o, lse) if return_lse else o


GEMV_NONE, GEMV_RMSNORM, GEMV_RELU2, GEMV_GATED = 0, 1, 2, 3


def gemv_takes(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Shapes tv_gemv_bf16_fwd is written for: 1..4 rows of bf16 against a bf16 (N, K) weight, f(x) within 128 KiB of LDS."""
    K = x.shape[-1]
    rows = x.numel() // max(K, 1)
    return (x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and weight.dim() == 2
            and 1 <= rows <= 4 and K % 8 == 0 and rows * K * 2 <= 128 * 1024 and weight.stride(1) == 1
            and weight.stride(0) % 8 == 0)


def gemv_fused(x, weight, bias=None, prologue=GEMV_NONE, delta=None, sum_out=None, norm_weight=None, eps=0.0,
               gate=None, group_size=0, conv=None, out_dtype=None):
    """y = f(x) @ weight.T (+ bias) for 1..4 rows — the linear layers of a decode step (torch.nn.Linear at q_len 1) with
    the operator in front of them computed in the kernel's prologue (several rows: mostly as a launch in front of a product on the matrix cores,
    see below): GEMV_RMSNORM (NemotronHRMSNorm with the
    block's residual add: `delta` is added to x first, the sum goes to `sum_out`), GEMV_RELU2 (the MLP activation),
    GEMV_GATED (MambaRMSNormGated with `gate`), rounding where the stand-alone operators round.
    `conv=(conv_state, weight, bias, row0)`: the outputs [row0, row0 + C) go through `causal_conv1d_update` (width 4,
    SiLU) on conv_state (B, C, 4) before they are stored — the mixer's in_proj -> conv pair as one launch (K < 8192).
    out_dtype fp32: the same values as fp32, from the product itself (GEMV_NONE, or one row's GEMV_RMSNORM without sum_out: a model's logits)."""
    if out_dtype is not None and out_dtype != x.dtype:
        if out_dtype != torch.float32 or gate is not None or conv is not None or sum_out is not None or prologue not in (GEMV_NONE, GEMV_RMSNORM):
            raise TimeViperHipError("gemv_fused: fp32 outputs of GEMV_NONE, or GEMV_RMSNORM without sum_out, only")
        if prologue == GEMV_NONE:
            delta = norm_weight = None
        elif norm_weight is None or x.numel() != x.shape[-1]:
            raise TimeViperHipError("gemv_fused: the norm in front of fp32 outputs is that of one row, with a weight")
        return _gemv_logits(x, weight, bias, delta, norm_weight, eps)
    _gpu(x, weight, bias, delta, sum_out, norm_weight, gate)
    K = x.shape[-1]
    x2 = _rows2d(x)
    M, N = x2.shape[0], weight.shape[0]
    if weight.shape[1] != K:
        raise TimeViperHipError(f"gemv_fused: weight {tuple(weight.shape)} against rows of {K}")
    # the C ABI carries no weight dtype: anything but dense bf16 rows would be re-interpreted silently
    if (x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or weight.stride(1) != 1 or weight.stride(0) % 8
            or K % 8):
        raise TimeViperHipError("gemv_fused: bf16 x and weight with dense rows of a multiple of 8 elements only "
                                f"(x {x.dtype}, weight {weight.dtype}, strides {tuple(weight.stride())}, K {K})")
    y = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    d2 = None if delta is None else _rows2d(delta)
    g2 = None if gate is None else _rows2d(gate)
    s2 = None if sum_out is None else sum_out.view(-1, K)
    for t in (d2, g2, s2):
        if t is not None and (t.shape != x2.shape or t.dtype != x.dtype):
            raise TimeViperHipError("gemv_fused: delta / gate / sum_out must have x's shape and dtype")
    if bias is not None and (bias.dtype != x.dtype or not bias.is_contiguous()):
        raise TimeViperHipError("gemv_fused: bias must be contiguous, of x's dtype")
    nw_dt = 0
    if norm_weight is not None:
        if not norm_weight.is_contiguous() or norm_weight.numel() != K:
            raise TimeViperHipError("gemv_fused: norm_weight must be a contiguous vector of K entries")
        nw_dt = _dt(norm_weight)
    cst = cw = cb = None
    row0 = nch = 0
    if conv is not None:
        cst, cw, cb, row0 = conv
        _gpu(cst, cw, cb)
        nch = cst.shape[1]
        if (cst.dtype != x.dtype or cw.dtype != x.dtype or not cst.is_contiguous() or not cw.is_contiguous()
                or cst.shape != (M, nch, 4) or cw.shape != (nch, 4) or (cb is not None and (cb.dtype != x.dtype or not cb.is_contiguous()))):
            raise TimeViperHipError("gemv_fused: conv needs a contiguous (rows, C, 4) state and (C, 4) weight of x's dtype")
    # (what the matrix-vector kernel refuses for one row it refuses for several: its bounds, not those of the launches that stand in for it)
    as_one = (M <= 4 and M * K * 2 <= 128 * 1024 and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0 and (conv is None or K < 8192)
              and (prologue != GEMV_RMSNORM or K <= 8192) and (prologue != GEMV_GATED or 0 < group_size <= 2048)
              and (norm_weight is None or norm_weight.data_ptr() % 16 == 0) and GEMV_NONE <= prologue <= GEMV_GATED)
    if as_one and rows_take(x2, weight) and (M > 2 or prologue == GEMV_NONE or N > K or N * K >= (1 << 23)):
        # several rows: the operator in front as its own launch and the product on the matrix cores, same rounding points.  us with the prologue
        # in the matrix-vector kernel | so, 2, 3 and 4 rows: 22 656 x 4 480, RMSNorm 37 41 45 | 35 35 35; 4 480 x 15 680, ReLU^2 30 43 49 | 25 25 25; 6 144 x
        # 2 048, RMSNorm 10.5 12.8 15.0 | 9.6 9.7 9.8; 1 024 x 1 024 without one 4.6 5.0 5.3 | 3.6 3.7 3.7.  Two rows of a small matrix
        # with few outputs do not pay for the launch (2 048 x 2 048, RMSNorm 7.0 | 7.1; 1 024 x 4 096, ReLU^2 6.5 | 7.0; 4 096 x 1 024, RMSNorm 7.2 | 6.7).
        f = _rows_prologue(x2, prologue, d2, s2, norm_weight, nw_dt, eps, g2, group_size, Kd=K)
        _rows_product(f, weight, bias, y, 0, cst, cw, cb, row0, nch)
        return y
    check(_capi.lib().tv_gemv_bf16_fwd(
        _p(x2), _p(weight), _p(bias), _p(y), M, N, K, x2.stride(0), weight.stride(0), N, int(prologue),
        _p(d2), 0 if d2 is None else d2.stride(0), _p(s2), 0 if s2 is None else s2.stride(0),
        _p(norm_weight), nw_dt, float(eps), _p(g2), 0 if g2 is None else g2.stride(0), int(group_size),
        _p(cst), _p(cw), _p(cb), int(row0), int(nch), _stream()), "tv_gemv_bf16_fwd")
    return y


ROWS_MAX = 32


def rows_weight(weight: torch.Tensor) -> bool:
    """Weights tv_gemm_rows_fwd reads: bf16 (N, K), K a multiple of 64, 16-byte aligned rows."""
    return (weight.dtype == torch.bfloat16 and weight.dim() == 2 and weight.shape[1] % 64 == 0 and weight.shape[1] > 0 and weight.stride(1) == 1
            and weight.stride(0) % 8 == 0 and weight.stride(0) < (1 << 24) and weight.data_ptr() % 16 == 0)


def rows_take(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Shapes tv_gemm_rows_fwd is written for: 2..32 rows of bf16 against such a weight."""
    Kd = x.shape[-1]
    n = x.numel() // max(Kd, 1)
    return x.is_cuda and x.dtype == torch.bfloat16 and 2 <= n <= ROWS_MAX and Kd % 64 == 0 and Kd > 0 and rows_weight(weight)


def rows_pay(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Shapes of `rows_take` on which tv_gemm_rows_fwd is faster than the library: more than 20 rows of a matrix of over 96 million entries
    are not (x, read again by every work-group, is then as many bytes as W; us, library | here: 131 072 x 4 480, 17 rows 198 | 189, 24: 199 | 207, 32: 198 |
    235; 65 536 x 4 480, 20: 102 | 98, 28: 102 | 108; 22 656 x 4 480, 24: 39 | 38, 32: 40 | 42; 15 680 x 4 480, 32: 37 | 29; 32 768 x 2 048, 32: 34 | 29)."""
    return rows_take(x, weight) and (x.numel() <= 20 * x.shape[-1] or weight.numel() <= 96_000_000)


def _rows_prologue(x2, prologue, d2, s2, norm_weight, nw_dt, eps, g2, group_size, Kd):
    """f(x) of gemv_fused for several rows, by the stand-alone kernels"""
    if prologue == GEMV_NONE:
        ok = x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and x2.stride(0) < (1 << 24) and x2.data_ptr() % 16 == 0
        return x2 if ok else x2.contiguous()
    if prologue not in (GEMV_RMSNORM, GEMV_RELU2, GEMV_GATED):
        raise TimeViperHipError(f"gemv_fused: prologue {prologue}")
    M = x2.shape[0]
    f = torch.empty((M, Kd), dtype=x2.dtype, device=x2.device)
    lib = _capi.lib()
    if prologue == GEMV_RELU2:
        xc = x2 if x2.is_contiguous() else x2.contiguous()
        check(lib.tv_relu2_fwd(_p(xc), _p(f), xc.numel(), _dt(xc), _stream()), "tv_relu2_fwd")
        return f
    if norm_weight is None or nw_dt not in (TV_F32, TV_BF16):
        raise TimeViperHipError("gemv_fused: norm weight (fp32 or bf16) needed")
    if prologue == GEMV_RMSNORM:
        check(lib.tv_rmsnorm_fwd(_p(x2), _p(d2), _p(norm_weight), _p(s2), _p(f), M, Kd, x2.stride(0),
                                 0 if d2 is None else d2.stride(0), 0 if s2 is None else s2.stride(0), Kd, float(eps), _dt(x2), nw_dt, _stream()),
              "tv_rmsnorm_fwd")
    else:
        check(lib.tv_rmsnorm_gated_fwd(_p(x2), _p(g2), _p(norm_weight), _p(f), M, Kd, int(group_size), x2.stride(0),
                                       0 if g2 is None else g2.stride(0), Kd, float(eps), _dt(x2), nw_dt, _stream()), "tv_rmsnorm_gated_fwd")
    return f


def _rows_product(f, weight, bias, y, epilogue=0, cst=None, cw=None, cb=None, row0=0, nch=0):
    N = weight.shape[0]
    y2 = y.view(-1, N)
    check(_capi.lib().tv_gemm_rows_fwd(_p(f), _p(weight), _p(bias), _p(y2), _dt(y2), f.shape[0], N, f.shape[1], f.stride(0), weight.stride(0),
                                       y2.stride(0), int(epilogue), _p(cst), _p(cw), _p(cb), int(row0), int(nch), _stream()), "tv_gemm_rows_fwd")


def _gemv_logits(x, weight, bias, delta, norm_weight, eps):
    _gpu(x, weight, bias, delta, norm_weight)
    x2 = _rows2d(x)
    N, Kd = weight.shape
    if not gemv_takes(x2, weight) or x2.shape[1] != Kd:
        raise TimeViperHipError(f"gemv_fused: 1..4 bf16 rows, got {tuple(x.shape)} {x.dtype} against {tuple(weight.shape)} {weight.dtype}")
    if bias is not None and (bias.dtype != x.dtype or not bias.is_contiguous() or bias.numel() != N):
        raise TimeViperHipError("gemv_fused: bias must be contiguous, of x's dtype")
    if x2.shape[0] > 1 and (x2.stride(0) % 8 or x2.data_ptr() % 16):
        x2 = x2.contiguous()
    if (delta is not None and (delta.dtype != x.dtype or delta.shape != x.shape or not delta.is_contiguous())) or (
            norm_weight is not None and (norm_weight.numel() != Kd or not norm_weight.is_contiguous())):
        raise TimeViperHipError("gemv_fused: a contiguous delta of x's shape and dtype, a contiguous norm weight")
    y = torch.empty(x.shape[:-1] + (N,), dtype=torch.float32, device=x.device)
    check(_capi.lib().tv_gemv_logits_fwd(_p(x2), _p(weight), _p(bias), _p(y), x2.shape[0], N, Kd, x2.stride(0), weight.stride(0), N, _p(delta), _p(norm_weight),
                                         0 if norm_weight is None else _dt(norm_weight), float(eps), _stream()), "tv_gemv_logits_fwd")
    return y


def rows_linear(x, weight, bias=None, relu2=False, conv=None, out_dtype=None, rounded=False):
    """x @ weight.T (+ bias) for 2..32 bf16 rows on the matrix cores (a decoded token for each of several sequences).  `relu2`: the squared
    ReLU of the bf16 product; `conv=(conv_state, weight, bias, row0)`: the outputs [row0, row0 + C) go through
    `causal_conv1d_update` (width 4, SiLU) on conv_state (rows, C, 4), as in `gemv_fused`.  out_dtype: bf16, or fp32 without either
    (`rounded`: of the bf16 values)."""
    if conv is None and out_dtype is None and not rounded and x.is_cuda and (r := _n.rows_linear(x, weight, bias, 1 if relu2 else 0)) is not None:
        return r
    _gpu(x, weight, bias)
    if not rows_take(x, weight) or weight.shape[1] != x.shape[-1]:
        raise TimeViperHipError(f"rows_linear: 2..{ROWS_MAX} bf16 rows of a multiple of 64 elements, got {tuple(x.shape)} against {tuple(weight.shape)}")
    if bias is not None and (bias.dtype != x.dtype or not bias.is_contiguous() or bias.numel() != weight.shape[0]):
        raise TimeViperHipError("rows_linear: bias must be contiguous, of x's dtype")
    x2 = _rows_prologue(_rows2d(x), GEMV_NONE, *(None,) * 7, Kd=x.shape[-1])
    cst = cw = cb = None
    row0 = nch = 0
    if conv is not None:
        cst, cw, cb, row0 = conv
        _gpu(cst, cw, cb)
        nch = cst.shape[1]
        if (cst.dtype != x.dtype or cw.dtype != x.dtype or not cst.is_contiguous() or not cw.is_contiguous() or cst.shape != (x2.shape[0], nch, 4)
                or cw.shape != (nch, 4) or (cb is not None and (cb.dtype != x.dtype or not cb.is_contiguous()))):
            raise TimeViperHipError("rows_linear: conv needs a contiguous (rows, C, 4) state and (C, 4) weight of x's dtype")
    y = torch.empty(x.shape[:-1] + (weight.shape[0],), dtype=out_dtype or x.dtype, device=x.device)
    _rows_product(x2, weight, bias, y, 1 if relu2 else 2 if rounded else 0, cst, cw, cb, row0, nch)
    return y


MID_MAX = 256


def mid_takes(x, weight, relu2=False) -> bool:
    """Products of up to 256 rows that tv_gemm_mid_fwd runs faster than the library (us, library | here):
      - any of at most 64 rows (15 680 x 4 480, 64 rows: 42 | 32; 1 024 x 4 480, 64: 21 | 10) but for 1, 2 or 3 x 4 096 outputs of a contraction no longer
        than they are (4 096 x 4 096, 48 rows: 13.5 | 14.3; 8 192 x 8 192: 32 | 36; 12 288 x 4 096: 25 | 29),
      - a long contraction into fewer outputs, 4 096 of them or more (4 480 x 15 680, 203 rows: 131 | 47; 4 480 x 5 120: 44 | 27; not 2 048 x 4 096, 96 rows:
        12.6 | 14.1, 256: 16 | 21),
      - 16 384 to 32 768 outputs from 80 rows on (22 656 x 4 480, 80 rows: 53 | 45, 128: 55 | 53, 203: 65 | 61, 256: 73 | 64; 32 768 x 4 480, 112: 84 | 62, 128: 64 | 64, 160: 67 | 68, 256: 79 | 76;
        16 384 x 4 096, 144: 42 | 50, 256: 54 | 50; over 25 such sizes .92 in the mean; 65 to 79 rows, .80 to .98 there, are still the library's).  Wider outputs are the library's (36 864 x 4 608:
        1.08 to 1.29 times as slow here, 50 304 x 4 480: 1.10 to 1.24, 65 536 x 4 096, 128 rows: 134 | 140), or
      - the squared ReLU into 4 096 outputs or more (its own pass saved; 15 680 x 4 480, with that pass, 96 rows 36 | 35, 160: 48 | 45, 203: 53 | 48, 256: 61 |
        52; prompts of these lengths wait for the host, where a launch less counts: 96 tokens 1 018 | 976 us a prompt of three such layers, 128: 1 005 | 975).
    Shorter contractions are the library's (6 144 x 2 048, 128 rows: 12 | 20)."""
    N, Kd = weight.shape if weight.dim() == 2 else (0, 0)
    n = x.numel() // max(x.shape[-1], 1)
    pays = (N >= 4096 and (N < Kd or relu2)) or (16384 <= N <= 32768 and n >= 80) or (n <= 64 and not (N % 4096 == 0 and Kd <= N <= 12288))
    return (pays and x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.shape[-1] == Kd and 2 <= n <= MID_MAX
            and Kd >= 4096 and Kd % 64 == 0 and N % 4 == 0 and weight.stride(1) == 1 and weight.stride(0) % 8 == 0
            and weight.stride(0) < (1 << 22) and weight.data_ptr() % 16 == 0)


def mid_before_rows(x, weight, relu2=False) -> bool:
    """Up to 32 rows of a prompt that `mid_linear` runs faster than `rows_linear`, whose work-groups read x again for every 32 rows of a large matrix: from 24 rows on of 45 million entries, from
    20 on of 60 to 140 million (us, rows_linear | mid_linear: 22 656 x 4 480: 16 rows 36.3 | 36.6, 20: 38.8 | 37.0, 32: 43.6 | 37.9; 15 680 x 4 480, 20: 28.4 | 28.0, 32: 30.2 | 27.6;
    4 480 x 15 680, 16: 30.4 | 30.6, 20: 34.1 | 29.9, 32: 35.5 | 31.0; 4 480 x 10 240, 24: 24.5 | 23.0, 32: 26.9 | 23.8; 9 216 x 5 120, 24: 25.4 | 23.0; over 105 such cases .93 in the mean; 20 rows of 11 016 x 4 480 1.04, of 24 576 x 6 144 1.17 times
    as slow).  Not where rows_linear's work-groups of 32 outputs fill .6 to 1 of a round, 4 865 to 8 192 outputs (24 rows: 6 144 x 8 192: 21.0 | 25.4, 7 168 x 7 168: 23.0 | 24.9, 8 192 x 8 192:
    27.7 | 29.9, 5 120 x 8 960: 21.9 | 23.1, 7 560 x 14 656: 43.0 | 42.3), nor smaller matrices or shorter contractions (4 480 x 5 120, 32: 15.0 | 16.4; 12 288 x 4 096: 23.3 | 28.2)."""
    N, Kd = weight.shape if weight.dim() == 2 else (0, 0)
    rows, entries = x.numel() // max(x.shape[-1], 1), weight.numel()
    pays = entries >= 45_000_000 if rows >= 24 else rows >= 20 and 60_000_000 <= entries <= 140_000_000
    return pays and Kd > 4096 and not 4864 < N <= 8192 and mid_takes(x, weight, relu2)


def large_takes(x, weight, relu2=False) -> bool:
    """Products of a long prompt that the persistent GEMM (tv_gemm_bf16_fwd) runs faster than the library: its 256 x 256 tiles are two
    rounds of the compute units or more and fill them, and
      - the output is wide, up to 12 288 rows (22 656 x 4 480, us, library | here: 1 500 rows, 70 % full, 355 | 275; 2 048: 445 | 319, 4 096: 726 | 617, 10 007: 1 494 |
        1 464; from there on the library's longer K loop wins: 14 000: 1 980 | 2 067, 80 000: 10 964 | 11 645, 163 940: 22 528 | 23 831),
      - the contraction is long, up to 32 768 rows (4 480 x 10 240: 6 011 rows 473 | 429, 10 007: 934 | 701, 28 000: 1 997 | 1 860, 40 000: 2 647 | 2 706, 163 940:
        10 637 | 10 797; 75 % full, 8 000 rows: 575 | 616; one round, 3 000: 191 | 195), or
      - the squared ReLU saves its own pass (15 680 x 4 480, with that pass: 2 048 rows 222 | 207, 10 007: 1 103 | 1 034, 163 940: 17 722 | 16 798).
    The rest stays the library's (15 680 x 4 480 alone; 12 288 x 4 096, 8 000 rows: 553 | 595)."""
    N, Kd = weight.shape if weight.dim() == 2 else (0, 0)
    rows = x.numel() // max(x.shape[-1], 1)
    tiles = -(-rows // 256) * -(-N // 256)
    if tiles <= CUS or rows <= MID_MAX or Kd < 4096:
        return False
    fill = tiles / (-(-tiles // CUS) * CUS)
    if relu2:
        pays = fill >= 0.75 and Kd <= 8192
    else:
        pays = (N >= 20480 and rows <= 12288 and fill >= 0.69) or (N < 20480 and Kd >= 8192 and rows <= 32768 and fill >= 0.8)
    return (pays and x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.shape[-1] == Kd and Kd % 128 == 0
            and N % 8 == 0 and 256 <= N < (1 << 22) and x.is_contiguous() and weight.is_contiguous() and x.data_ptr() % 16 == 0
            and weight.data_ptr() % 16 == 0 and gemm_persist_on())


GEMM_GLU = 5


def small_linear(x, weight, bias=None, epilogue: int = GEMM_BIAS, out=None, tile: int = 0):
    """`linear_fused` on small tiles (tv_gemm_small_fwd): x (rows, K) bf16, weight (N, K); GEMM_GLU: the two halves of weight's rows, `glu_linear`'s result"""
    if x.is_cuda and (r := _n.small_linear(x, weight, bias, epilogue, out, tile)) is not None:
        return r
    _gpu(x, weight, bias, out)
    N, Kd = weight.shape
    if epilogue == GEMM_GLU:
        N //= 2
    if x.dtype != torch.bfloat16 or weight.dtype != x.dtype or x.dim() != 2 or x.shape[1] != Kd or x.stride(1) != 1 or weight.stride(1) != 1:
        raise TimeViperHipError(f"small_linear: {tuple(x.shape)} {x.dtype} against {tuple(weight.shape)}")
    if out is None:
        if epilogue == GEMM_ACCUM:
            raise TimeViperHipError("small_linear: GEMM_ACCUM needs `out`")
        out = x.new_empty((x.shape[0], N))
    if out.shape != (x.shape[0], N) or out.dtype != x.dtype or out.stride(1) != 1:
        raise TimeViperHipError("small_linear: `out` must be (rows, N) of x's dtype")
    if bias is not None and (bias.dtype not in (torch.float32, torch.bfloat16) or not bias.is_contiguous() or bias.numel() != weight.shape[0]):
        raise TimeViperHipError("small_linear: bias must be contiguous, fp32 or bf16")
    check(_capi.lib().tv_gemm_small_fwd(_p(x), _p(weight), None if epilogue == GEMM_ACCUM else _p(bias), _p(out), x.shape[0], N, Kd, x.stride(0),
                                        weight.stride(0), out.stride(0), int(epilogue), TV_F32 if bias is None else _dt(bias), tile, _stream()),
          "tv_gemm_small_fwd")
    return out


def small_tile(rows: int, n: int, k: int, glu: bool = False) -> int:
    """The tile of tv_gemm_small_fwd for rows x n outputs (of either factor with `glu`) where it replaces a library call of a short forward, -1 where it does not.
    Such a forward waits for the host, which a library call takes 19 us of and this one 8: some sizes take longer on the device than the library's, which shows where
    the device is busy with other work or the calls are captured.  64 x 64 up to 1.2 rounds of the compute units (two of them run on one), up to two in contractions of more
    than 2 048 columns (at most 4 608, at most 1 536 rows), else 64 x 128 up to 1.3, 128 x 128 up to two; tv_gemm_small_fwd takes the next larger tile where one of the first two
    is more than a round and that one fits.
    us on the device, weights out of cache, library | here: 64 x 64: 1 152 x 1 152, 729 rows: 12.5 | 8.0; 1 152 x 4 352, 729: 22 | 18; 64 x 128: 1 152 x 1 152, 1 458: 13.7 | 10.8;
    1 152 x 4 352, 1 458: 31 | 26; 128 x 128: 3 456 x 1 152, 729: 17.9 | 14.0; 5 120 x 2 048, 729: 26 | 23; two rounds, 3 456 x 1 152, 1 458: 19 | 24, 2 187: 29 | 26; 5 120 x 2 048, 1 458: 34 | 40."""
    if not 2 <= rows <= 2304 or n < 512 or k % 64 or (k > 2048 and (k > 4608 or rows > 1536)):
        return -1
    over = lambda tm, tn: -(-rows // tm) * -(-n * (2 if glu else 1) // tn)
    if over(64, 64) <= CUS * 6 // 5:
        return 3
    if k > 2048:
        return 3 if over(64, 64) <= CUS * 2 else -1
    if over(64, 128) <= CUS * 4 // 3:
        return 2
    if over(128, 128) <= CUS:
        return 0
    return 1 if over(128, 128) <= CUS * 2 else -1


def round_takes(x, weight) -> bool:
    """Rows beyond `small_tile` on which 128 x 128 tiles (tile 0 of `small_linear`) are faster on the device than the library: one round of them, at least 60 % full, 53 from
    3 072 columns on, 66 of less than 1 024 outputs; outputs wider than a contraction of 2 816 columns and more are the library's.  us with weights out of cache, library (adding to its output) |
    here: 1 152 x 4 352: 1 499 rows (42 %): 31 | 33, 1 883 (53 %): 36 | 33, 2 395: 40 | 33, 3 419: 43 | 37; 1 152 x 1 152: 2 139 (60 %): 13.0 | 12.7, 2 395: 15.3 | 12.7, 2 651: 13.4 | 13.1, 3 547:
    15.4 | 15.6; 1 024 x 4 096: 1 755 (44 %): 27 | 29, 2 139: 35 | 29, 4 059: 41 | 35; 1 408 x 6 144: 1 243 (43 %): 40 | 45, 1 499: 50 | 43, 2 779: 59 | 51; 2 048 x 2 048: 987 (50 %): 17.1 | 18.4, 1 243:
    22 | 19; 4 096 x 2 048, 603: 23 | 20, 987: 25.6 | 24.1.  As shares of the library's time: 768 x 3 072: 3 456 rows (63 %) 1.03, 3 763 (70 %): .89, 5 376: .83; 6 144 x 4 096, 307 - 640 rows 1.31 -
    1.03, 8 192 x 3 072, 307: 1.10, 9 216 x 3 072, 179: 1.34, 10 240 x 4 096, 384: 1.20.  Two rounds are the library's (1 152 x 4 352, 3 645: 45 | 59)."""
    rows, (n, k) = x.shape[0], weight.shape
    tiles = -(-rows // 128) * -(-n // 128)
    full = 66 if n < 1024 else 53 if k >= 3072 else 60
    return (full * CUS <= 100 * tiles <= 100 * CUS and (n <= k or k < 2816) and n >= 512 and n % 8 == 0 and 1024 <= k <= 6144 and k % 64 == 0
            and products_take(x, weight))


def tail_plan(rows: int, n: int, k: int):
    """(work-groups a tile, whole tiles in front) for a product whose last round of 256 x 256 tiles is at most 46 % full (half from 12 288 columns on): those tiles
    share the compute units, as many work-groups each as fit (us, one work-group a tile | here: 22 656 x 4 480, 1 400 rows, 2.09 rounds, 276 | 237, 3 000: 475 | 457,
    2 500, 48 %: 386 | 393; 4 480 x 15 680, 4 096: 569 | 409, 5 000: 592 | 508); None where it is fuller, or where there is a single round or a short contraction."""
    tiles = -(-rows // 256) * -(-n // 256)
    last = tiles % CUS
    if tiles <= CUS or not 0 < last <= (CUS // 2 if k > 12288 else CUS * 46 // 100) or k < 4096 or k % 64 or n % 4:
        return None
    return min(CUS // last, 16), tiles - last


def split_takes(x, weight, relu2=False):
    """Products of more than 256 rows that tv_gemm_split_fwd runs faster than the library, and that `large_takes` does not have: (work-groups a tile, whole tiles in
    front of those), None where the product is not one of them.  Over 260 drawn sizes that the rule takes (outputs 4 096 - 30 000, columns 4 096 - 24 000, multiples of 64, rows 257 -
    16 000, weights out of cache) a factor of 1.30 in the mean; the library's own times jump with its choice of a kernel, and 2 in 100 of the sizes lose 4 - 6 % to a
    good one (us, library | here):
      - a long contraction into fewer outputs whose tiles leave half of the compute units idle: as many work-groups a tile as fit one round, if they fill 80 % of
        it, more than two up to 8 192 columns (4 480 x 10 240: 300 rows 59 | 52, 512: 85 | 59, 1 024: 108 | 90, 1 536: 137 | 124; 4 480 x 15 680: 300: 92 | 67, 512: 137 | 75,
        1 400: 349 | 177; 75 % full, 600 rows of 8 192 x 28 672: 254 | 287; two of 8 192 x 8 192: 800: 107 | 113, 1 024: 117 | 120; two, 44 % without the padding, 13 312 x 18 432, 280: 186 | 200),
      - a contraction longer than the outputs whose last round is 80 % full (75 from 12 288 columns on): one work-group a tile; in a first round (75 % without the
        padding: 9 088 x 12 800, 1 335 rows, 72: 238 | 259) and in contractions of less than 8 192 only at widths that the library's 256 columns do not divide (4 096 x 11 008, 3 900 rows:
        227 | 237; 5 376 x 5 632, 8 835: 354 | 364; 7 680 x 8 064, 9 993: 817 | 889; 4 480 x 15 680, an
        odd number of steps: 3 000 rows 532 | 306, 10 007: 1 382 | 999, 14 000: 1 728 | 1 360; 4 480 x 10 240: 3 000: 219 | 203; 4 480 x 5 120: 3 000: 117 | 107, 6 011:
        224 | 207), not two rounds that are full, where the library is in step (7 000 x 15 680: 654 | 680),
      - several rounds of which the last is nearly empty (`tail_plan`), of outputs up to 1.25 times as wide as the contraction is long, from more than 4 096 columns on (4 096 x 4 096,
        5 000 rows: 135 | 139), or of 20 480 and more up to 12 288 rows and eight rounds (21 440 x 11 840, 9 244, twelve: 3 191 | 3 327), unless a fifth of the rows would be padding
        (28 672 x 8 192, 600: 259 | 268) (22 656 x 4 480: 768 rows 182 | 132, 2 200: 378 | 339; 4 480 x 10 240: 3 700: 464 | 248, 8 192: 561 | 527; 5 120 x 4 480: 3 400:
        149 | 130, 7 000: 382 | 241; 4 480 x 5 120, 4 096: 167 | 148, 5 000: 184 | 182),
      - the squared ReLU in a single round that is 72 % full, 63 without the padding (12 288 x 4 096, 800 rows, 59: 77 | 84; 28 672 x 8 192, 300, 51: 157 | 179), or in several with such
        a last one (15 680 x 4 480, with the pass that it saves: 700 rows 101 | 90, 1 024: 122 | 103, 1 400: 185 | 170, 2 200: 266 | 243)."""
    N, Kd = weight.shape if weight.dim() == 2 else (0, 0)
    rows = x.numel() // max(x.shape[-1], 1)
    tiles = -(-rows // 256) * -(-N // 256)
    if rows <= MID_MAX or N < 4096 or Kd < 4096 or rows > 32768:
        return None
    fill = tiles / (-(-tiles // CUS) * CUS)
    fit, useful = CUS // tiles, rows * N / 65536           # (useful: tiles without the padding)
    plan = None
    if fit >= 2:
        pays = not relu2 and N <= Kd and Kd >= 8192 and fit <= 8 and tiles * fit >= 0.8 * CUS and (fit > 2 or (Kd > 8192 and 2 * useful >= 0.65 * CUS))
        plan = (fit, 0) if pays else None
    elif tiles <= CUS:
        pays = fill >= 0.72 and useful >= 0.63 * CUS and Kd <= 8192 if relu2 else fill >= 0.8 and useful >= 0.75 * CUS and N <= Kd and N % 256 != 0
        plan = (1, 0) if pays else None
    elif relu2:
        plan = tail_plan(rows, N, Kd) if Kd <= 8192 else None
    else:
        padded = rows < 0.8 * 256 * -(-rows // 256) and tiles % CUS > CUS // 8
        if (4 * N <= 5 * Kd and Kd > 4096) or (N >= 20480 and rows <= 12288 and tiles <= 8 * CUS and not padded):
            plan = tail_plan(rows, N, Kd)
        in_step = tiles <= 2 * CUS and fill > 0.96
        if plan is None and N < Kd and fill >= (0.75 if Kd > 12288 else 0.8) and (
                (Kd % 128 != 0 and not in_step) if Kd >= 8192 else N % 256 != 0):
            plan = (1, 0)
    takes = (plan and x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and x.shape[-1] == Kd and Kd % 64 == 0 and N % 4 == 0
             and Kd < (1 << 22) and x.is_contiguous() and weight.is_contiguous() and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)
    return plan if takes and gemm_persist_on() and not large_takes(x, weight, relu2) else None


def split_linear(x, weight, bias=None, relu2=False, splits=1, full=0):
    """x @ weight.T (+ bias, then the squared ReLU of the bf16 product) on tiles of 256 x 256 outputs, `splits` work-groups a tile but for the first `full`."""
    if x.is_cuda and (r := _n.split_linear(x, weight, bias, relu2, splits, full)) is not None:
        return r
    _gpu(x, weight, bias)
    N, Kd = weight.shape
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or x.shape[-1] != Kd or weight.stride(1) != 1:
        raise TimeViperHipError(f"split_linear: bf16 rows of {Kd} elements, got {tuple(x.shape)} {x.dtype} against {weight.dtype}")
    if bias is not None and (bias.dtype not in (torch.float32, torch.bfloat16) or not bias.is_contiguous() or bias.numel() != N):
        raise TimeViperHipError("split_linear: bias must be contiguous, fp32 or bf16")
    x2 = _rows2d(x)
    y = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    lib, M = _capi.lib(), x2.shape[0]
    need = int(lib.tv_gemm_split_workspace_bytes(M, N, splits, full))
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    check(lib.tv_gemm_split_fwd(_p(x2), _p(weight), _p(bias), _p(y), M, N, Kd, x2.stride(0), weight.stride(0), N, 3 if relu2 else 0,
                                TV_F32 if bias is None else _dt(bias), splits, full, _p(ws), need, _stream()), "tv_gemm_split_fwd")
    return y


def mid_linear(x, weight, bias=None, relu2=False):
    """x @ weight.T (+ bias, then the squared ReLU of the bf16 product) for up to 256 bf16 rows (a short prompt)."""
    if x.is_cuda and (r := _n.mid_linear(x, weight, bias, relu2)) is not None:
        return r
    _gpu(x, weight, bias)
    N, Kd = weight.shape
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or x.shape[-1] != Kd:
        raise TimeViperHipError(f"mid_linear: bf16 rows of {Kd} elements, got {tuple(x.shape)} {x.dtype} against {weight.dtype}")
    if bias is not None and (bias.dtype != x.dtype or not bias.is_contiguous() or bias.numel() != N):
        raise TimeViperHipError("mid_linear: bias must be contiguous, of x's dtype")
    x2 = _rows2d(x)
    if x2.stride(1) != 1 or x2.stride(0) % 8 or x2.stride(0) >= (1 << 22) or x2.data_ptr() % 16:
        x2 = x2.contiguous()
    if bias is not None and bias.data_ptr() % 8:
        bias = bias.clone()
    y = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    lib, M = _capi.lib(), x2.shape[0]
    need = int(lib.tv_gemm_mid_workspace_bytes(M, N, Kd))
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    check(lib.tv_gemm_mid_fwd(_p(x2), _p(weight), _p(bias), _p(y), M, N, Kd, x2.stride(0), weight.stride(0), N, 1 if relu2 else 0, _p(ws), need, _stream()),
          "tv_gemm_mid_fwd")
    return y


def mid_linears_take(x, weights, pays: bool = True) -> bool:
    """Whether `mid_linears` is there for these matrices and (pays) faster than one product after the other: the three projections of an attention layer for a short
    prompt's rows ((5 120, 1 024, 1 024) x 4 480, us, a launch each (up to 32 rows tv_gemm_rows_fwd, the library) | one: 2 rows 21 | 17, 24: 28 | 18, 64: 39 | 21, 128: 66 | 29, 203: 66 | 32,
    256: 85 | 35; (2 048, 2 048, 2 048) x 4 096, 16 rows 21 | 16, 100: 38 | 24, 256: 47 | 30; over 18 sets of 3 584 to 24 576 outputs and 4 096 to 16 384 columns .4 to .98).  Up to 16 rows not
    where every one of them has more than 32 million entries: they fill the chip one by one (three of 6 144 x 6 144, 2 rows 1.12 times as slow, 16: 1.03)."""
    Kd = x.shape[-1]
    n = x.numel() // max(Kd, 1)
    return (2 <= n <= MID_MAX and Kd >= 4096 and Kd % 64 == 0 and x.is_cuda and x.dtype == torch.bfloat16 and 2 <= len(weights) <= 3
            and sum([w.shape[0] for w in weights]) >= 4096 and (not pays or n > 16 or min([w.shape[0] for w in weights]) * Kd <= 32_000_000)
            and all([w.dtype == torch.bfloat16 and w.dim() == 2 and w.shape[1] == Kd and w.shape[0] % 4 == 0 and w.shape[0] > 0 and w.stride(1) == 1
                     and w.stride(0) % 8 == 0 and Kd <= w.stride(0) < (1 << 22) and w.data_ptr() % 16 == 0 for w in weights]))


def mid_linears(x, weights):
    """[x @ w.T for w in weights] for two or three matrices and up to 256 bf16 rows, in one launch (shapes: `mid_linears_take`, whether it pays or not)."""
    if x.is_cuda and len(weights) == 3 and (r := _n.mid_linears(x, *weights)) is not None:
        return r
    _gpu(x, *weights)
    if not mid_linears_take(x, weights, pays=False):
        raise TimeViperHipError(f"mid_linears: 2..{MID_MAX} bf16 rows against two or three matrices, got {tuple(x.shape)} against {[tuple(w.shape) for w in weights]}")
    x2 = _rows2d(x)
    if x2.stride(1) != 1 or x2.stride(0) % 8 or x2.stride(0) >= (1 << 22) or x2.data_ptr() % 16:
        x2 = x2.contiguous()
    ys = [torch.empty(x.shape[:-1] + (w.shape[0],), dtype=x.dtype, device=x.device) for w in weights]
    n, lib, M, Kd = len(weights), _capi.lib(), x2.shape[0], x2.shape[1]
    ptrs = lambda ts: (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])
    N = (ctypes.c_int * n)(*[w.shape[0] for w in weights])
    ldw, ldy = (ctypes.c_int64 * n)(*[w.stride(0) for w in weights]), (ctypes.c_int64 * n)(*N)
    need = int(lib.tv_gemm_mid_multi_workspace_bytes(M, N, n, Kd))
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    check(lib.tv_gemm_mid_multi_fwd(_p(x2), ptrs(weights), ptrs(ys), N, n, M, Kd, x2.stride(0), ldw, ldy, _p(ws), need, _stream()), "tv_gemm_mid_multi_fwd")
    return ys


def kv_append(k, v, k_cache, v_cache, pos) -> None:
    """k_cache[:, pos] = k[:, 0], v_cache[:, pos] = v[:, 0] for (B, 1, H, D) keys and values and an int64 position on the device (both
    caches' `index_copy_` in one launch)."""
    B, one, H, D = k.shape
    size = k.element_size()
    ok = (k.is_cuda and one == 1 and k.dtype == v.dtype == k_cache.dtype == v_cache.dtype and k.shape == v.shape and k_cache.shape == v_cache.shape
          and k_cache.shape[0] == B and k_cache.shape[2:] == k.shape[2:] and (H * D * size) % 16 == 0 and pos.dtype == torch.int64 and pos.numel() == 1
          and all([t.stride(3) == 1 and t.stride(2) == D and not (t.data_ptr() | t.stride(0) * size | t.stride(1) * size) % 16
                   for t in (k, v, k_cache, v_cache)]))
    if not ok:
        k_cache.index_copy_(1, pos, k)
        v_cache.index_copy_(1, pos, v)
        return
    _gpu(k, v, k_cache, v_cache, pos)
    st = lambda t, d: t.stride(d) * size
    check(_capi.lib().tv_kv_append(_p(k), _p(v), _p(k_cache), _p(v_cache), _p(pos), B, k_cache.shape[1], H * D * size, st(k, 0), st(v, 0), st(k_cache, 0),
                                   st(k_cache, 1), st(v_cache, 0), st(v_cache, 1), _stream()), "tv_kv_append")


_plan_streams = {}            # device -> the stream that `step_plan` launches on


def _plan_stream(device):
    """tv_step_plan_stream's of the device, which is the current one"""
    side = _plan_streams.get(device)
    if side is None:
        made = ctypes.c_void_p()
        check(_capi.lib().tv_step_plan_stream(ctypes.byref(made)), "tv_step_plan_stream")
        side = _plan_streams.setdefault(device, torch.cuda.ExternalStream(made.value, device=device))
    return side


def step_plan(starts, slots, counts, capacity: int, device):
    """int32 device tensors of a packed step (cache.StepPlan): cu, start, slot, rows, seq, keys and, one token per sequence, the (3, B) tensor
    behind start, rows and keys (else None for these two).  One launch, on a stream of its own: the tensors are complete when the call returns, for
    every stream, and nothing waits for what the current one still has to do (unless both share one of the device's hardware queues).  Their memory is kept for the current stream as for any tensor; a step that runs on another one
    says so (`SlotStateCache.commit`)."""
    B, T = len(starts), sum(counts)
    if torch.cuda.is_current_stream_capturing():
        raise TimeViperHipError("step_plan: the numbers of a step do not belong into a captured graph (plan the step first)")
    single = B == T
    up = lambda n: (n + 3) & ~3                                   # 16-byte aligned parts
    sizes = [3 * B if single else T, B + 1, B, T] + ([] if single else [B])
    now = torch.cuda.current_stream(device)
    side = _plan_stream(now.device)
    with torch.cuda.stream(side):
        buf = torch.empty((sum(up(n) for n in sizes),), dtype=torch.int32, device=device)
    _gpu(buf)
    buf.record_stream(now)                                        # (memory of the side stream: not given out again before `now` has left it)
    parts, at = [], 0
    for n in sizes:
        parts.append(buf[at:at + n])
        at += up(n)
    if single:
        moving, (_, cu, slot, seq) = parts[0].view(3, B), parts
        start, rows, keys = moving
    else:
        moving, keys, (rows, cu, slot, seq, start) = None, None, parts
    ints = ctypes.c_int * B
    check(_capi.lib().tv_step_plan(ints(*starts), ints(*slots), ints(*counts), B, capacity, _p(cu), _p(start), _p(slot), _p(rows), _p(seq), _p(keys),
                                   side.cuda_stream), "tv_step_plan")
    side.synchronize()
    return cu, start, slot, rows, seq, keys, moving


def count_up(pos, lens) -> None:
    """pos += 1 (int64, one entry), lens += 1 (int32), in one launch on the GPU"""
    if not (pos.is_cuda and lens.is_cuda and pos.dtype == torch.int64 and pos.numel() == 1 and lens.dtype == torch.int32 and lens.is_contiguous()):
        pos += 1
        lens += 1
        return
    _gpu(pos, lens)
    check(_capi.lib().tv_count_up(_p(pos), _p(lens), lens.numel(), _stream()), "tv_count_up")


def argmax_rows(x, count=None):
    """x.argmax(-1) of the fp32 logits of up to 65 535 rows.  count=(pos, lens): `count_up` of them in the same launch (pos may be None)."""
    pos, lens = count or (None, None)
    takes = x.is_cuda and x.dim() == 2 and x.dtype == torch.float32 and x.stride(1) == 1 and 0 < x.shape[0] <= 65535 and 8192 <= x.shape[1] <= (1 << 30)
    if count and not (takes and lens.dtype == torch.int32 and lens.is_contiguous() and lens.is_cuda
                      and (pos is None or pos.is_cuda and pos.dtype == torch.int64 and pos.numel() == 1)):
        out = argmax_rows(x)
        if pos is None:
            lens += 1
        else:
            count_up(pos, lens)
        return out
    if not takes:
        return x.argmax(-1)
    _gpu(x, pos, lens)
    lib, B = _capi.lib(), x.shape[0]
    out = torch.empty((B,), dtype=torch.int64, device=x.device)
    ws = torch.empty((int(lib.tv_argmax_rows_workspace_bytes(B)),), dtype=torch.uint8, device=x.device)
    check(lib.tv_argmax_rows_count(_p(x), _p(out), B, x.shape[1], x.stride(0), _p(pos), _p(lens), lens.numel() if count else 0, _p(ws), ws.numel(), _stream()),
          "tv_argmax_rows_count")
    return out


def _decode_attn_takes(q, k, v) -> bool:
    """Shapes tv_attn_decode_fwd is written for (the rest stays on tv_flash_attn_fwd with one query row)."""
    return (q.dtype == torch.bfloat16 and q.shape[-1] == 128 and k.shape[1] >= 256
            and os.environ.get("TV_ATTN_DECODE", "1") != "0"
            and all(s % 8 == 0 for t in (q, k, v) for s in t.stride()[:3])
            and all(t.data_ptr() % 16 == 0 for t in (q, k, v)))


def flash_attn_decode(q, k, v, seqlens_k=None, softmax_scale=None, return_lse=False, out=None):
    """One query token per sequence against a K / V cache: q (B, 1, Hq, 128) bf16, k / v (B, Lk, Hkv, 128) ->
    (B, 1, Hq, 128) (the q_len == 1 call of modeling_nano.py:1198-1209).  `seqlens_k`: int32 tensor (B,) ON THE GPU with
    the keys in use per sequence (<= Lk, the capacity of the cache buffers) — the form a captured decode step replays
    with; None: all Lk keys."""
    _gpu(q, k, v, seqlens_k)
    B, Lq, Hq, D = q.shape
    Lk, Hkv = k.shape[1], k.shape[2]
    if Lq != 1:
        raise TimeViperHipError("flash_attn_decode: one query token per sequence")
    if seqlens_k is not None and (seqlens_k.dtype != torch.int32 or seqlens_k.numel() != B or not seqlens_k.is_contiguous()):
        raise TimeViperHipError("flash_attn_decode: seqlens_k must be a contiguous int32 tensor of `batch` entries")
    fix = lambda t: t if t.stride(-1) == 1 else t.contiguous()
    q, k, v = fix(q), fix(k), fix(v)
    scale = 1.0 / math.sqrt(D) if softmax_scale is None else float(softmax_scale)
    o = torch.empty((B, 1, Hq, D), dtype=q.dtype, device=q.device) if out is None else out
    if o.shape != (B, 1, Hq, D) or o.dtype != q.dtype or o.stride(-1) != 1:
        raise TimeViperHipError("flash_attn_decode: out must be (B, 1, Hq, D) of q's dtype with unit last stride")
    lse = torch.empty((B, Hq, 1), dtype=torch.float32, device=q.device) if return_lse else None
    lib = _capi.lib()
    ws = torch.empty((max(int(lib.tv_attn_decode_workspace_bytes(B, Hq, Hkv, Lk)), 16),), dtype=torch.uint8,
                     device=q.device)
    check(lib.tv_attn_decode_fwd(
        _p(q), _p(k), _p(v), _p(o), _p(lse), B, Lk, _p(seqlens_k), Hq, Hkv, D,
        q.stride(0), q.stride(2), k.stride(0), k.stride(1), k.stride(2),
        v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(2),
        scale, _dt(q), _p(ws), ws.numel() * ws.element_size(), _stream()), "tv_attn_decode_fwd")
    return (o, lse) if return_lse else o


def _flash_attention_forward(query_states, key_states, value_states, attention_mask=None,
                             query_length=None, is_causal=True, dropout=0.0, position_ids=None,
                             softmax_scale=None, sliding_window=None, use_top_left_mask=False,
                             **kwargs):
    """transformers' helper as NemotronHFlashAttention2 calls it (:1198-1209)."""
    if attention_mask is not None or sliding_window is not None:
        raise TimeViperHipError("_flash_attention_forward: padding mask / sliding window unsupported")
    causal = is_causal and not (use_top_left_mask and query_states.shape[1] == 1)
    return flash_attn_func(query_states, key_states, value_states, dropout,
                           softmax_scale=softmax_scale, causal=causal)


def scaled_dot_product_attention(query, key, value, attn_mask=None, dropout_p=0.0,
                                 is_causal=False, scale=None):
    """F.scaled_dot_product_attention layout: (B, H, L, D) in and out."""
    if attn_mask is not None:
        raise TimeViperHipError("scaled_dot_product_attention: attn_mask unsupported")
    o = flash_attn_func(query.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2),
                        dropout_p, softmax_scale=scale, causal=is_causal)
    return o.transpose(1, 2)


def flash_attn_varlen_qkvpacked_func(qkv, cu_seqlens, max_seqlen, dropout_p=0.0,
                                     softmax_scale=None, causal=False, **kwargs):
    """qkv (nnz, 3, H, D), sequences [cu_seqlens[i], cu_seqlens[i+1]) (flash_attention_class.py:59-66, :68-91).
    Equal lengths — what the InternVideo2 ViT produces: every clip has the same token count — are ONE launch over
    a (nseq, len) view; a ragged batch (the `key_padding_mask` / `unpad_input` path of the reference) runs one launch per
    run of consecutive equal-length sequences.  The boundaries are read on the host: one device-to-host copy of
    `cu_seqlens` when it lives on the GPU (the reference's unpad_input synchronises for max_seqlen as well)."""
    nnz, three, H, D = qkv.shape
    assert three == 3
    nseq = cu_seqlens.numel() - 1
    if nseq > 0 and nnz == nseq * max_seqlen:                # equal lengths: no host read
        x = qkv.view(nseq, max_seqlen, 3, H, D)
        o = flash_attn_func(x[:, :, 0], x[:, :, 1], x[:, :, 2], dropout_p, softmax_scale, causal)
        return o.reshape(nnz, H, D)
    cu = [int(v) for v in cu_seqlens.tolist()]
    if cu[0] != 0 or cu[-1] != nnz or any(b < a for a, b in zip(cu, cu[1:])):
        raise TimeViperHipError("flash_attn_varlen_qkvpacked_func: cu_seqlens must rise from 0 to nnz")
    out = torch.empty((nnz, H, D), dtype=qkv.dtype, device=qkv.device)
    i = 0
    while i < nseq:
        n = cu[i + 1] - cu[i]
        j = i + 1
        while j < nseq and cu[j + 1] - cu[j] == n:
            j += 1
        if n > 0:
            x = qkv[cu[i]:cu[j]].view(j - i, n, 3, H, D)
            out[cu[i]:cu[j]] = flash_attn_func(x[:, :, 0], x[:, :, 1], x[:, :, 2], dropout_p, softmax_scale,
                                               causal).reshape((j - i) * n, H, D)
        i = j
    return out


# --------------------------------------------------------------- token ops
def gather_rows(src: torch.Tensor, index: torch.Tensor) -> torch.Tensor:
    """dst[r] = src[index[r]] for a (rows, D) tensor; index int64 on the GPU."""
    _gpu(src, index)
    s2 = _rows2d(src)
    idx = index.to(torch.int64).contiguous()
    out = torch.empty((idx.numel(), s2.shape[1]), dtype=src.dtype, device=src.device)
    check(_capi.lib().tv_gather_rows(_p(s2), _p(idx), _p(out), idx.numel(), s2.shape[1],
                                     s2.stride(0), out.stride(0), _dt(src), _stream()),
          "tv_gather_rows")
    return out


def uniform_keep_indices(n_tokens: int, keep: int, offset: int = 0, device="cuda"):
    """torch.linspace(0, n-1, keep, dtype=long) with CPU semantics, + offset
    (modeling_nano.py:1946-1957), produced on the GPU, bit-exact."""
    out = torch.empty((keep,), dtype=torch.int64, device=device)
    check(_capi.lib().tv_uniform_keep_indices(_p(out), int(n_tokens), int(keep), int(offset),
                                              _stream()), "tv_uniform_keep_indices")
    return out


def dropped_indices(keep_sorted: torch.Tensor, start: int, n: int) -> torch.Tensor:
    """[start, start+n) minus keep_sorted, ascending (modeling_nano.py:1966-1970)."""
    _gpu(keep_sorted)
    ks = keep_sorted.to(torch.int64).contiguous()
    out = torch.empty((n - ks.numel(),), dtype=torch.int64, device=ks.device)
    check(_capi.lib().tv_dropped_indices(_p(ks), ks.numel(), int(start), int(n), _p(out),
                                         _stream()), "tv_dropped_indices")
    return out


def attn_rank_scores(q_row: torch.Tensor, k: torch.Tensor, n_keys: int, vis_start: int,
                     n_vis: int, scale: Optional[float] = None) -> torch.Tensor:
    """Importance of each vision token for pdrop "attn" (modeling_nano.py:1914-1939):
    q_row (Hq, D) = last prompt token's queries, k (L, Hkv, D); softmax over keys
    [0, n_keys) per head in fp32, mean over heads, slice [vis_start, vis_start+n_vis)."""
    _gpu(q_row, k)
    Hq, D = q_row.shape
    L, Hkv, _ = k.shape
    q_row = q_row.contiguous()
    if k.stride(-1) != 1:
        k = k.contiguous()
    scale = 1.0 / math.sqrt(D) if scale is None else float(scale)
    lib = _capi.lib()
    ws_bytes = lib.tv_attn_rank_workspace_bytes(int(n_keys), Hq)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=k.device)
    scores = torch.empty((n_vis,), dtype=torch.float32, device=k.device)
    check(lib.tv_attn_rank_scores(_p(q_row), _p(k), _p(scores), int(n_keys), Hq, Hkv, D,
                                  k.stride(0), k.stride(1), int(vis_start), int(n_vis), scale,
                                  _dt(k), _p(ws), ws_bytes, _stream()), "tv_attn_rank_scores")
    return scores


def attn_rank_logits(q_row: torch.Tensor, k: torch.Tensor, scale: Optional[float] = None) -> torch.Tensor:
    """First half of `attn_rank_scores` for a sequence shard: logits (n_keys, Hq) fp32 of this
    rank's keys k (n_keys, Hkv, D) against the broadcast query row, with the reference's roundings."""
    _gpu(q_row, k)
    Hq, D = q_row.shape
    n, Hkv, _ = k.shape
    q_row = q_row.contiguous()
    if k.stride(-1) != 1:
        k = k.contiguous()
    scale = 1.0 / math.sqrt(D) if scale is None else float(scale)
    out = torch.empty((n, Hq), dtype=torch.float32, device=k.device)
    check(_capi.lib().tv_attn_rank_logits(_p(q_row), _p(k), _p(out), int(n), Hq, Hkv, D, k.stride(0),
                                          k.stride(1), scale, _dt(k), _stream()), "tv_attn_rank_logits")
    return out


def attn_rank_scores_from_logits(logits: torch.Tensor, vis_start: int, n_vis: int, dtype) -> torch.Tensor:
    """Second half: softmax over ALL keys per head, mean over heads (roundings in `dtype`, the
    activation dtype), slice [vis_start, vis_start + n_vis).  logits (n_keys, Hq) fp32."""
    _gpu(logits)
    logits = logits.contiguous()
    n, Hq = logits.shape
    ws = torch.empty(2 * Hq, dtype=torch.float32, device=logits.device)
    scores = torch.empty((n_vis,), dtype=torch.float32, device=logits.device)
    check(_capi.lib().tv_attn_rank_scores_from_logits(_p(logits), _p(scores), int(n), Hq, int(vis_start),
                                                      int(n_vis), _DT[dtype], _p(ws), ws.numel() * 4,
                                                      _stream()), "tv_attn_rank_scores_from_logits")
    return scores


# ---------------------------------------------------------------- patch embed
def apply_rotary_pos_emb_(q, k, cos, sin):
    """In-place rotary embedding of q (B, L, Hq, D) and k (B, L, Hkv, D) (views with a
    contiguous head dim) with cos / sin (B, L, D): modeling_qwen2.py:89-113."""
    _gpu(q, k, cos, sin)
    B, L, _, D = q.shape
    cs = cos.to(q.dtype).reshape(B * L, D).contiguous()
    sn = sin.to(q.dtype).reshape(B * L, D).contiguous()
    for t in (q, k):
        assert t.stride(-1) == 1 and (B == 1 or t.stride(0) == L * t.stride(1))
        check(_capi.lib().tv_rope_fwd(_p(t), _p(cs), _p(sn), B * L, t.shape[2], D, t.stride(1),
                                      t.stride(2), _dt(t), _stream()), "tv_rope_fwd")
    return q, k


def silu_mul(gate, up):
    """silu(gate) * up over the last dim (Qwen2MLP, modeling_qwen2.py:78-80)."""
    _gpu(gate, up)
    g2, u2 = _rows2d(gate), _rows2d(up)
    y = torch.empty(g2.shape, dtype=gate.dtype, device=gate.device)
    check(_capi.lib().tv_silu_mul_fwd(_p(g2), _p(u2), _p(y), g2.shape[0], g2.shape[1], g2.stride(0),
                                      u2.stride(0), y.stride(0), _dt(gate), _stream()), "tv_silu_mul_fwd")
    return y.view(gate.shape)


def tome_merge_round(x, size, r: int, heads: int = 16):
    """One ToMe round for every frame (tome.py:14-83): x (F, T, C), size (F, T, 1) or None ->
    (x' (F, T-r, C), size' (F, T-r, 1)); rows = [kept even tokens, descending match score |
    odd tokens with their merged partners], size-weighted average."""
    _gpu(x, size)
    F_, T, Cc = x.shape
    x = x.contiguous()
    sz = None if size is None else size.reshape(F_, T).to(x.dtype).contiguous()
    xo = torch.empty((F_, T - r, Cc), dtype=x.dtype, device=x.device)
    so = torch.empty((F_, T - r, 1), dtype=x.dtype, device=x.device)
    lib = _capi.lib()
    ws_bytes = lib.tv_tome_workspace_bytes(F_, T, Cc, heads)
    ws = torch.empty(max(int(ws_bytes), 16), dtype=torch.uint8, device=x.device)
    check(lib.tv_tome_merge_round(_p(x), _p(sz), _p(xo), _p(so), F_, T, Cc, heads, int(r), _dt(x),
                                  _p(ws), int(ws_bytes), _stream()), "tv_tome_merge_round")
    return xo, so


def patch_embed(pixels, weight, bias=None, pos=None, patch: Optional[int] = None):
    """pixels (F, C, H, W) -> (F, gh*gw, Dout); weight is the Conv2d weight
    (Dout, C, p, p) (or Conv3d (Dout, C, 1, p, p)); pos (gh*gw, Dout) optional."""
    _gpu(pixels, weight, bias, pos)
    F_, Cin, H, W = pixels.shape
    Dout = weight.shape[0]
    p = int(weight.shape[-1]) if patch is None else int(patch)
    pixels = pixels.contiguous()
    w = weight.reshape(Dout, -1).to(pixels.dtype).contiguous()
    assert w.shape[1] == Cin * p * p
    b = None if bias is None else bias.to(pixels.dtype).contiguous()
    ps = None if pos is None else pos.reshape(-1, Dout).to(pixels.dtype).contiguous()
    out = torch.empty((F_, (H // p) * (W // p), Dout), dtype=pixels.dtype, device=pixels.device)
    ws = torch.empty((_capi.lib().tv_patch_embed_workspace_bytes(Dout, Cin, p),), dtype=torch.uint8,
                     device=pixels.device)
    check(_capi.lib().tv_patch_embed_fwd(_p(pixels), _p(w), _p(b), _p(ps), _p(out), F_, Cin, H,
                                         W, p, Dout, _dt(pixels), _p(ws), _stream()),
          "tv_patch_embed_fwd")
    return out


def patch_embed_video(pixels, weight, bias=None, pos=None):
    """Conv3d k=s=(1,p,p) on (B, C, T, H, W) -> (B, T*gh*gw, Dout), token order
    (t, py, px) as vit_scale_clean.py:455-460."""
    _gpu(pixels, weight, bias, pos)
    B, Cin, T, H, W = pixels.shape
    Dout, p = weight.shape[0], int(weight.shape[-1])
    pixels = pixels.contiguous()
    w = weight.reshape(Dout, -1).to(pixels.dtype).contiguous()
    b = None if bias is None else bias.to(pixels.dtype).contiguous()
    ps = None if pos is None else pos.reshape(-1, Dout).to(pixels.dtype).contiguous()
    npatch = (H // p) * (W // p)
    out = torch.empty((B, T * npatch, Dout), dtype=pixels.dtype, device=pixels.device)
    ws = torch.empty((_capi.lib().tv_patch_embed_workspace_bytes(Dout, Cin, p),), dtype=torch.uint8,
                     device=pixels.device)
    check(_capi.lib().tv_patch_embed_strided_fwd(
        _p(pixels), _p(w), _p(b), _p(ps), _p(out), B * T, Cin, H, W, p, Dout, T,
        Cin * T * H * W, H * W, T * H * W, _dt(pixels), _p(ws), _stream()), "tv_patch_embed_strided_fwd")
    return out


# ------------------------------------------------- post-norm models on a 32-bit residual stream
def _vec(t: torch.Tensor, n: int, what: str) -> torch.Tensor:
    if t.numel() != n or not t.is_contiguous():
        raise TimeViperHipError(f"{what}: a contiguous vector of {n} entries is needed, got {tuple(t.shape)}")
    return t


def _i32(t: Optional[torch.Tensor], n: int, what: str) -> None:
    if t is not None and (t.dtype != torch.int32 or t.numel() < n or not t.is_contiguous()):
        raise TimeViperHipError(f"{what}: a contiguous int32 tensor of {n} entries is needed")


def rms_norm_ex(x, weight, eps, weight_offset=0.0, gate=None, residual=None, mult=1.0, out_dtype=None, sum_out=None,
                y2=None, y2_rows=None, need_y=True):
    """n = x / sqrt(mean(x^2) + eps) * (weight_offset + weight) over the last dim [, * sigmoid(gate)].  With `residual` (fp32):
    s = residual + mult * n; returns (y, s) with y = s in `out_dtype` (default: the weight's).  Without: returns n.
    `y2` / `y2_rows`: the result rows are written to rows y2_rows of the 2-D buffer y2 as well (a cache)."""
    _gpu(x, weight, gate, residual, sum_out, y2, y2_rows)
    x2 = _rows2d(x)
    rows, D = x2.shape
    _vec(weight, D, "rms_norm_ex weight")
    yd = out_dtype or weight.dtype
    g2 = None if gate is None else _rows2d(gate)
    r2 = s2 = None
    if gate is not None and (gate.dtype != weight.dtype or g2.shape != x2.shape):
        raise TimeViperHipError("rms_norm_ex: gate must have x's shape and the weight's dtype")
    if residual is not None:
        r2 = _rows2d(residual)
        if residual.dtype != torch.float32 or r2.shape != x2.shape:
            raise TimeViperHipError("rms_norm_ex: the residual is fp32 and has x's shape")
        s2 = torch.empty((rows, D), dtype=torch.float32, device=x.device) if sum_out is None else _rows2d(sum_out)
        if s2.dtype != torch.float32 or s2.shape != x2.shape:
            raise TimeViperHipError("rms_norm_ex: sum_out is fp32 and has x's shape")
    y = torch.empty((rows, D), dtype=yd, device=x.device) if need_y else None
    if y2 is not None:
        _i32(y2_rows, rows, "rms_norm_ex y2_rows")
        if y2.dtype != yd or y2.dim() != 2 or y2.shape[1] != D or y2.stride(1) != 1:
            raise TimeViperHipError("rms_norm_ex: y2 is a (rows, D) buffer of the output dtype")
    st = lambda t: 0 if t is None else t.stride(0)
    check(_capi.lib().tv_rmsnorm_ex_fwd(
        _p(x2), _p(weight), _p(g2), _p(r2), _p(s2), _p(y), _p(y2), _p(y2_rows), st(y2), rows, D, x2.stride(0), st(g2), st(r2), st(s2),
        st(y), float(eps), float(mult), float(weight_offset), _dt(x), _dt(weight), _DT[yd], _stream()), "tv_rmsnorm_ex_fwd")
    y = None if y is None else y.view(x.shape)
    return y if residual is None else (y, s2.view(x.shape))


def moe_combine_norm(expert_out, pos, weights, residual, norm_weight, eps, weight_offset=0.0, mult=1.0, out_dtype=None):
    """u = sum_j weights[:, j] * expert_out[pos[:, j]] (pos < 0: the residual row, an identity expert), then as `rms_norm_ex` with
    this residual.  Returns (y, s)."""
    _gpu(expert_out, pos, weights, residual, norm_weight)
    rows, D = residual.shape
    top = pos.shape[1]
    _i32(pos, rows * top, "moe_combine_norm pos")
    _vec(norm_weight, D, "moe_combine_norm weight")
    if (residual.dtype != torch.float32 or residual.stride(1) != 1 or weights.dtype != torch.float32 or not weights.is_contiguous()
            or weights.shape != pos.shape or expert_out.shape[1] != D or expert_out.stride(1) != 1):
        raise TimeViperHipError("moe_combine_norm: fp32 residual (rows, D), fp32 weights (rows, top), expert rows of D elements")
    yd = out_dtype or norm_weight.dtype
    y = torch.empty((rows, D), dtype=yd, device=residual.device)
    s = torch.empty((rows, D), dtype=torch.float32, device=residual.device)
    check(_capi.lib().tv_moe_combine_norm_fwd(
        _p(expert_out), _p(pos), _p(weights), top, _p(residual), _p(norm_weight), _p(s), _p(y), rows, D, expert_out.stride(0),
        residual.stride(0), s.stride(0), y.stride(0), float(eps), float(mult), float(weight_offset), _dt(expert_out),
        _dt(norm_weight), _DT[yd], _stream()), "tv_moe_combine_norm_fwd")
    return y, s


def embed_scaled(ids, table, scale=1.0, positions=None, plan=None, need_h=True):
    """(fp32 rows, rows in the table's dtype) of `table[ids] * scale`; ids int64 on the GPU.  `positions` (max, D): the row of the
    token's place in its sequence is added (plan: the step's `cache.StepPlan`; its places lie within the table)."""
    _gpu(ids, table, positions)
    flat = ids.reshape(-1).contiguous()
    V, D = table.shape
    if flat.dtype != torch.int64 or not table.is_contiguous():
        raise TimeViperHipError("embed_scaled: int64 ids and a contiguous table")
    x = torch.empty((flat.numel(), D), dtype=torch.float32, device=table.device)
    h = torch.empty((flat.numel(), D), dtype=table.dtype, device=table.device) if need_h else None
    seq = cu = start = None
    if positions is not None:
        seq, cu, start = _plan(plan, flat.numel(), "embed_scaled")[:3]
        if positions.dtype != table.dtype or positions.dim() != 2 or positions.shape[1] != D or not positions.is_contiguous():
            raise TimeViperHipError("embed_scaled: positions (max, D) of the table's dtype")
    check(_capi.lib().tv_embed_scaled_fwd(_p(flat), _p(table), _p(x), _p(h), flat.numel(), D, V, float(scale), _p(positions), _p(seq), _p(cu),
                                          _p(start), 0 if positions is None else positions.shape[0], _dt(table), _stream()),
          "tv_embed_scaled_fwd")
    return x, h


# ------------------------------------------------- parallel layers on a 32-bit residual stream
def _plan(plan, rows, what):
    """(seq, cu, start, slot) of a step's plan for `rows` packed rows"""
    B = len(plan.slots)
    if plan.rows.numel() != rows:
        raise TimeViperHipError(f"{what}: {rows} rows in a step of {plan.rows.numel()}")
    for t, n in ((plan.seq, rows), (plan.cu, B + 1), (plan.start, B), (plan.slot, B)):
        _gpu(t)
        _i32(t, n, what + " plan")
    return plan.seq, plan.cu, plan.start, plan.slot


def _shift_state(state, plan, D, what):
    """(slots, 2, D) fp32 blocks, possibly one layer's slice of a wider state: the distance between two blocks"""
    if (state.dtype != torch.float32 or state.dim() != 3 or state.shape[1:] != (2, D) or state.stride(2) != 1 or state.stride(1) != D
            or max(plan.slots) >= state.shape[0]):
        raise TimeViperHipError(f"{what}: a (slots, 2, {D}) fp32 state with dense blocks")
    return state.stride(0)


def norm_shift(x, gain, eps, pending=None, pending_weight=None, shift=None, state=None, plan=None, need_h=True):
    """x (T, D) fp32 -> (x', h, hs): x' = x + rms(pending) * pending_weight (x itself without `pending`), h = rms(x') * gain (a tensor of one
    element), hs = h + (h_before - h) * shift with the h of the sequence's previous token (`state` (slots, 2, D) fp32, advanced in
    place; None without `shift`).  h and hs have the gain's dtype."""
    if x.is_cuda:
        steps = (None,) * 5 + (0, False) if plan is None else (plan.seq, plan.cu, plan.start, plan.slot, plan.rows, max(plan.slots, default=0), plan.decode)
        if (r := _n.norm_shift(x, gain, eps, pending, pending_weight, shift, state, *steps, need_h)) is not None:
            return r
    _gpu(x, gain, pending, pending_weight, shift, state)
    T, D = x.shape
    if x.dtype != torch.float32 or not x.is_contiguous() or gain.numel() != 1:
        raise TimeViperHipError("norm_shift: dense fp32 rows and a gain of one element")
    xo, ps = None, 0
    if pending is not None:
        if pending.shape != x.shape or pending.dtype != gain.dtype or pending.stride(1) != 1 or pending_weight.dtype != gain.dtype:
            raise TimeViperHipError("norm_shift: pending rows and weight of x's width and the gain's dtype")
        _vec(pending_weight, D, "norm_shift pending weight")
        xo, ps = torch.empty_like(x), pending.stride(0)
    h = torch.empty((T, D), dtype=gain.dtype, device=x.device) if need_h or shift is None else None
    hs, seq, cu, start, slot, sst = None, None, None, None, None, 0
    if shift is not None:
        _vec(shift, D, "norm_shift shift")
        if shift.dtype != gain.dtype:
            raise TimeViperHipError("norm_shift: shift of the gain's dtype")
        hs = torch.empty((T, D), dtype=gain.dtype, device=x.device)
        seq, cu, start, slot = _plan(plan, T, "norm_shift")
        sst = _shift_state(state, plan, D, "norm_shift")
    check(_capi.lib().tv_norm_shift_fwd(
        _p(x), _p(pending), _p(pending_weight), _p(xo), _p(gain), _p(shift), _p(state if shift is not None else None), _p(seq), _p(cu), _p(start), _p(slot),
        _p(h), _p(hs), T, D, ps, sst, float(eps), int(plan is not None and plan.decode), _dt(gain), _stream()), "tv_norm_shift_fwd")
    return x if xo is None else xo, h, hs


def residual_add(x, u):
    """(x + u in fp32, its rounding to u's dtype); x (T, D) fp32"""
    if x.is_cuda and (r := _n.residual_add(x, u)) is not None:
        return r
    _gpu(x, u)
    if x.dtype != torch.float32 or not x.is_contiguous() or u.shape != x.shape or u.stride(1) != 1:
        raise TimeViperHipError("residual_add: dense fp32 x and u of its shape")
    xo, h = torch.empty_like(x), torch.empty(x.shape, dtype=u.dtype, device=x.device)
    check(_capi.lib().tv_residual_add_fwd(_p(x), _p(u), _p(xo), _p(h), x.shape[0], x.shape[1], u.stride(0), _dt(u), _stream()),
          "tv_residual_add_fwd")
    return xo, h


ACT_SIGMOID, ACT_GELU_TANH = 0, 1


def products_take(x, *weights) -> bool:
    """What the products below need of a layer's rows and matrices: bf16 on the GPU, whole 16-byte rows, no gradients, no autocast, plain tensors."""
    return (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.stride(0) < (1 << 22) and x.data_ptr() % 16 == 0
            and x.shape[0] > 0 and not torch.is_grad_enabled() and not torch.is_autocast_enabled()
            and all(type(w) in (torch.Tensor, torch.nn.Parameter) and w.dtype == torch.bfloat16 and w.dim() == 2 and w.stride(1) == 1 and w.stride(0) % 8 == 0
                    and 64 <= w.stride(0) < (1 << 22) and w.data_ptr() % 16 == 0 for w in weights))


def bias_takes(b) -> bool:
    """What the products below need of a bias: bf16 in whole 16-byte pieces, or none (the library takes any address)"""
    return b is None or (type(b) in (torch.Tensor, torch.nn.Parameter) and b.dtype == torch.bfloat16 and b.is_contiguous() and b.data_ptr() % 16 == 0)


def small_takes(x, weight, glu: bool = False, most: int = 2304, bias=None) -> int:
    """`small_tile` of x (rows, K) against weight, -1 where the rows are more than `most` or the operands are not what the kernel reads"""
    n = weight.shape[0] // 2 if glu else weight.shape[0]
    tile = small_tile(x.shape[0], n, x.shape[1], glu) if x.shape[0] <= most else -1
    reach = ((n if glu else 0) + 128) * weight.stride(0) < (1 << 30)             # (both halves of a gated pair at 32-bit offsets)
    return tile if tile >= 0 and n % 8 == 0 and reach and products_take(x, weight) and bias_takes(bias) else -1


def glu_takes(x, weight, bias=None, waits: bool = True) -> bool:
    """Rows on which `glu_linear` takes the place of the library's product and the pass over it.  waits: the caller waits for its launches, which is worth 20 us of the
    device: tiles (256 rows x 128 outputs) for half of a first round, or 65 % of several, or a few rows behind rounds that are nine tenths full that go to small tiles
    (`glu_lead`), in contractions of 2 048 or less.  Else it has to be the faster one: 60 % of a round without the padding, 70 % of several
    (60 in contractions of 2 048 or less), up to 6 144 columns.
    us, two launches | here: 2 x 5 632 x 2 048: 512 rows, 34 % full, 38 | 44; 600: 39 | 45, 700: 51 | 45, 1 000: 62 | 49; 1 300, 52 % of two rounds: 75 | 89; 1 800, 69 %: 95 | 90;
    3 000: 146 | 136, 4 000: 186 | 146, 6 011: 301 | 230, 8 192: 405 | 285; with small tiles, 1 403: 73 | 72; 2 x 7 680 x 2 048, 1 147: 96 | 74; 2 x 4 096 x 1 024, 2 098: 53 | 47;
    2 x 8 192 x 3 072: 300, half full, 47 | 69, 600: 66 | 72, 1 400: 135 | 140; 2 x 11 008 x 4 096: 300: 75 | 89, 900: 170 | 173; 2 x 14 336 x 4 096, 700: 165 | 174; 2 x 28 672 x 8 192, 1 800:
    1 269 | 1 306, 6 011: 3 870 | 3 978."""
    N, Kd, rows = weight.shape[0] // 2, weight.shape[1], x.shape[0]
    tiles = -(-rows // 256) * -(-N // 128)
    if not (rows >= 256 and N >= 2048 and N % 8 == 0 and Kd >= 1024 and Kd % 128 == 0 and tiles >= CUS // 2):
        return False
    rounds, lead = -(-tiles // CUS), (rows, -1)
    pays = tiles <= CUS or tiles >= 0.65 * CUS * rounds
    if pays and not waits:
        pays = rows * N >= (0.6 if rounds == 1 or Kd <= 2048 else 0.7) * 32768 * CUS * rounds and Kd <= 6144
    if not pays and Kd <= 2048:
        lead = glu_lead(rows, N)
        pays = lead[1] == 0 and lead[0] // 256 * -(-N // 128) >= 0.9 * CUS * (tiles // CUS)
    return pays and products_take(x, weight) and bias_takes(bias) and gemm_persist_on()


def glu_lead(rows: int, n: int):
    """(rows in front that fill whole rounds of tv_gemm_glu_fwd's tiles, the tile of tv_gemm_small_fwd for the rows behind them); (rows, -1): one launch for all.
    128 x 128 small tiles: one a compute unit, or two to a third of them (us, one launch | two, 2 x 5 632 x 2 048: 1 536 rows 90 | 73, 2 939: 138 | 123, 3 196, 264 small
    tiles, 139 | 131, 6 011: 235 | 222; 2 x 4 096 x 1 024: 4 476: 85 | 78, 4 736, 320: 84 | 83; 2 x 11 008 x 4 096: 2 171: 341 | 307, 3 072, 344: 433 | 424)."""
    wide = -(-n // 128)
    rounds = -(-rows // 256) * wide // CUS
    lead = rounds * CUS // wide * 256
    small = -(-(rows - lead) // 128) * -(-n // 64)
    if rounds < 1 or not 256 <= lead < rows or small > CUS * 4 // 3:
        return rows, -1
    return lead, 0 if small <= CUS else 1


def glu_linear(x, weight, bias, out):
    """out = gelu_tanh(x @ Wg.T + bg) * (x @ Wu.T + bu) for the two halves of weight's rows and of the bias, on tv_gemm_glu_fwd, the rows behind its whole
    rounds on tv_gemm_small_fwd (`glu_lead`); fp32 until the one rounding."""
    _gpu(x, weight, bias, out)
    N, Kd = weight.shape[0] // 2, weight.shape[1]
    if (x.dtype != torch.bfloat16 or weight.dtype != x.dtype or out.dtype != x.dtype or weight.shape[0] % 2 or x.shape[1] != Kd or x.stride(1) != 1
            or weight.stride(1) != 1 or out.stride(1) != 1 or out.shape != (x.shape[0], N)):
        raise TimeViperHipError(f"glu_linear: {tuple(x.shape)} bf16 against {tuple(weight.shape)} into {tuple(out.shape)}")
    _bf16_bias(bias, 2 * N, "glu_linear")
    lead, tile = glu_lead(x.shape[0], N) if (N + 128) * weight.stride(0) < (1 << 30) else (x.shape[0], -1)       # (the small tiles reach both halves at 32-bit offsets)
    check(_capi.lib().tv_gemm_glu_fwd(_p(x), _p(weight), _p(bias), _p(out), lead, N, Kd, x.stride(0), weight.stride(0), out.stride(0), _stream()),
          "tv_gemm_glu_fwd")
    if tile >= 0:
        check(_capi.lib().tv_gemm_small_fwd(_p(x[lead:]), _p(weight), _p(bias), _p(out[lead:]), x.shape[0] - lead, N, Kd, x.stride(0), weight.stride(0),
                                            out.stride(0), GEMM_GLU, _dt(bias), tile, _stream()), "tv_gemm_small_fwd")
    return out


def split_add_takes(x, weight, bias=None, waits: bool = True) -> int:
    """Work-groups a tile with which tv_gemm_split_add_fwd takes the place of the library's product and the pass that adds it, 0 where it does not.  waits: the caller
    waits for its launches: a contraction of 4 096 columns or more whose tiles, shared, fill 75 % of one round, 16 work-groups a tile at most.  Else it has to be the
    faster one: contractions of 7 168 columns or more, shares of more than 768, 65 % of the round without the padding; or a single row of tiles (64 rows
    or more of 256) in 16 shares of 704 columns or more.
    us, two launches | here: 2 048 x 7 680: 40 rows 17 | 20, 256: 26 | 30, 512: 30 | 39, 700: 41 | 42, 1 100: 55 | 53, 1 400: 55 | 58, 2 500: 92 | 84, 4 000: 130 | 121; whole
    tiles, 6 011: 160 | 168; 1 024 x 5 120: 256: 16 | 28, 1 800: 38 | 41, 6 011: 72 | 77; 1 536 x 5 632, 1 800: 45 | 51; 3 072 x 11 264: 70: 40 | 28, 203: 40 | 37, 300, 55 % full, 42 | 47, 400: 59 | 49,
    1 100: 111 | 86; 4 096 x 15 104: 17: 28 | 32, 203: 62 | 47, 700: 115 | 93, 1 800: 218 | 195; 8 192 x 36 864, 600, 59 % full: 344 | 379."""
    N, Kd = weight.shape
    rows = x.shape[0]
    tiles = -(-rows // 256) * -(-N // 256)
    splits = min(CUS // tiles, 16, Kd // 192) if tiles else 0
    pays = splits >= 2 and (tiles * splits >= 0.75 * CUS or splits == 16) and Kd >= 4096 and Kd % 64 == 0 and N >= 1024 and N % 4 == 0
    if pays and not waits:
        pays = Kd >= 7168 and ((Kd > 768 * splits and rows * N * splits >= 0.65 * 65536 * CUS) or (splits == 16 and 64 <= rows <= 256 and Kd >= 704 * 16))
    return splits if pays and products_take(x, weight) and bias_takes(bias) else 0


@functools.lru_cache(maxsize=1024)
def small_add_plan(rows: int, n: int, k: int):
    """(tile of `small_linear`, splits) on which tv_gemm_small_add_fwd adds a product of long contraction and few outputs to the residual stream, None where
    tv_gemm_split_add_fwd or the library is faster: weights of at most 2^24 entries, at least two splits of 128 x 128 tiles in one round of the compute units.
    us, the library and the pass that adds | 256 x 256 tiles | here: 2 048 x 7 680: 64 rows 26 | 22 | 17, 256: 31 | 33 | 23, 300: 37 | 34 | 27, 512: 38 | 39 | 31, 900: 49 | 47 | 44, 1 100, one split,
    69 | 53 | 62; 1 024 x 5 120: 100: 14 | 19 | 12, 512: 19 | 28 | 17, 2 000: 41 | 42 | 33; 1 536 x 5 632: 17: 11 | 16 | 12, 300: 23 | 28 | 18, 1 100: 43 | 40 | 34; 2 048 x 4 096: 40: 12 | 17 |
    12, 256: 19 | 27 | 16; larger matrices, 3 072 x 11 264: 40: 31 | 27 | 27, 300: 52 | 46 | 49.  More than 768 rows of more than 9 000 columns are one split's march, longer than the 256 x 256
    tiles' shares: 1 536 x 10 240, 900 rows 1.06 times their time, 1 024 x 16 384, 1 300: 1.13, 2 000: 1.09 (768: .96; 1 456 x 5 632, 1 024: .89).
    The choice is the least of an estimate in us (a step of 64 columns, more where more work-groups stream; a split's sums written and read), a fit to those sizes with 17
    to 2 000 rows: .1 % slower in the mean than the best choice, 2.5 % at most."""
    if n * k > 1 << 24 or k < 4096 or n < 1024 or (rows > 768 and k > 9000) or -(-rows // 128) * -(-n // 128) * 2 > CUS:
        return None
    best = None
    for tile, tm, tn, step, more in ((3, 64, 64, .166, .042), (2, 64, 128, .248, .074), (0, 128, 128, .334, .174)):
        tiles = -(-rows // tm) * -(-n // tn)
        for splits in range(1, min(8, CUS // tiles, k // 256) + 1):
            t = -(-(k // 64) // splits) * (step + more * tiles * splits / CUS) + splits * (.195 + 1.38e-6 * rows * n)
            if best is None or t < best[0]:
                best = (t, tile, splits)
    return best[1:] if best else None


def small_add_takes(x, weight, bias=None):
    """`small_add_plan` of x (rows, K) against weight, None where the operands are not what the kernel reads"""
    plan = small_add_plan(x.shape[0], *weight.shape) if x.shape[0] > 0 else None
    return plan if plan and weight.shape[0] % 8 == 0 and weight.shape[1] % 64 == 0 and products_take(x, weight) and bias_takes(bias) else None


def small_add_linear(x, weight, residual, bias=None, tile=3, splits=1):
    """(residual + x @ weight.T (+ bias) in fp32, its bf16 copy) on small tiles whose contraction is split (`small_add_plan`)"""
    if x.is_cuda and (r := _n.small_add_linear(x, weight, residual, bias, tile, splits)) is not None:
        return r
    _gpu(x, weight, residual, bias)
    N, Kd = weight.shape
    if (x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or x.shape[1] != Kd or x.stride(1) != 1 or weight.stride(1) != 1 or residual.dtype != torch.float32
            or residual.shape != (x.shape[0], N) or not residual.is_contiguous()):
        raise TimeViperHipError(f"small_add_linear: {tuple(x.shape)} bf16 against {tuple(weight.shape)} onto {tuple(residual.shape)} fp32")
    if bias is not None:
        _bf16_bias(bias, N, "small_add_linear")
    lib, M = _capi.lib(), x.shape[0]
    res, h = torch.empty_like(residual), torch.empty((M, N), dtype=x.dtype, device=x.device)
    need = int(lib.tv_gemm_small_add_workspace_bytes(M, N, splits))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=x.device)
    check(lib.tv_gemm_small_add_fwd(_p(x), _p(weight), _p(bias), _p(residual), _p(res), _p(h), M, N, Kd, x.stride(0), weight.stride(0), int(tile), int(splits),
                                    _p(ws), need, _stream()), "tv_gemm_small_add_fwd")
    return res, h


def split_add_linear(x, weight, residual, bias=None, splits=1):
    """(residual + x @ weight.T (+ bias) in fp32, its bf16 copy): `split_linear` with the residual stream behind it"""
    if x.is_cuda and (r := _n.split_add_linear(x, weight, residual, bias, splits)) is not None:
        return r
    _gpu(x, weight, residual, bias)
    N, Kd = weight.shape
    if (x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or x.shape[1] != Kd or x.stride(1) != 1 or weight.stride(1) != 1 or residual.dtype != torch.float32
            or residual.shape != (x.shape[0], N) or not residual.is_contiguous()):
        raise TimeViperHipError(f"split_add_linear: {tuple(x.shape)} bf16 against {tuple(weight.shape)} onto {tuple(residual.shape)} fp32")
    if bias is not None:
        _bf16_bias(bias, N, "split_add_linear")
    lib, M = _capi.lib(), x.shape[0]
    res, h = torch.empty_like(residual), torch.empty((M, N), dtype=x.dtype, device=x.device)
    need = int(lib.tv_gemm_split_workspace_bytes(M, N, splits, 0))
    ws = torch.empty(need, dtype=torch.uint8, device=x.device) if need else None
    check(lib.tv_gemm_split_add_fwd(_p(x), _p(weight), _p(bias), _p(residual), _p(res), _p(h), M, N, Kd, x.stride(0), weight.stride(0), TV_BF16, splits, 0,
                                    _p(ws), need, _stream()), "tv_gemm_split_add_fwd")
    return res, h


def side_takes(h, table, gate, proj, waits: bool = True) -> bool:
    """Shapes tv_token_side_fwd is written for: a side of 128 columns.  Where the caller does not wait for its launches, rows on which it is faster than the three of
    them, too: its work-groups read the first matrix whole, so that few rows of a wide model take half as long as thousands (us, three launches | here, 512 wide: 17 to
    8 192 rows 12 - 18 | 8 - 11; 1 024: 12 - 23 | 9 - 16; 2 048: 40 rows 12 | 16, 1 000: 14 | 14, 2 000: 17 | 20, 2 048: 17 | 18, 2 200: 25 | 20, 3 000: 23 | 21, 6 011: 28 | 26; 3 072: 4 000: 30 | 34, 6 011: 46 | 35;
    4 096: 203: 15 | 24, 5 000: 42 | 44, 6 011: 50 | 45; 8 192: 203: 16 | 76, 6 011: 69 | 79)."""
    rows, width = h.shape[0], gate.shape[1]
    return (gate.shape[0] == 128 and width % 32 == 0 and table.stride(0) % 4 == 0
            and (waits or width <= 1024 or (width <= 2048 and rows > 2048) or (width <= 4096 and rows >= 6000))
            and products_take(h, gate, proj) and table.data_ptr() % 8 == 0 and table.dtype == torch.bfloat16 and table.stride(1) == 1)


def token_side(h, ids, table, gate, proj):
    """proj @ (gelu_tanh(gate @ h) * table[ids]) for the rows of h in one launch (tv_token_side_fwd); ids are checked where the step was planned"""
    if h.is_cuda and (r := _n.token_side(h, ids, table, gate, proj)) is not None:
        return r
    _gpu(h, ids, table, gate, proj)
    T, D = h.shape
    S = gate.shape[0]
    if (any(t.dtype != torch.bfloat16 or t.stride(1) != 1 for t in (h, table, gate, proj)) or gate.shape != (S, D) or proj.shape != (D, S) or table.shape[1] != S
            or ids.dtype != torch.int64 or ids.numel() != T or not ids.is_contiguous()):
        raise TimeViperHipError(f"token_side: rows {tuple(h.shape)} with {tuple(gate.shape)}, {tuple(proj.shape)} and a table {tuple(table.shape)}")
    y = torch.empty((T, D), dtype=h.dtype, device=h.device)
    check(_capi.lib().tv_token_side_fwd(_p(h), _p(ids), _p(table), _p(gate), _p(proj), _p(y), T, D, S, table.shape[0], h.stride(0), table.stride(0),
                                        gate.stride(0), proj.stride(0), D, _stream()), "tv_token_side_fwd")
    return y


def gated_mul(a, b, act, ids=None, out=None):
    """f(a) * b over rows, f = sigmoid or the tanh form of gelu; `ids` (int64): row r meets b[ids[r]].  `out`: rows to write to."""
    if a.is_cuda and (r := _n.gated_mul(a, b, act, ids, out)) is not None:
        return r
    _gpu(a, b, ids, out)
    T, n = a.shape
    o = torch.empty((T, n), dtype=a.dtype, device=a.device) if out is None else out
    if (b.dtype != a.dtype or b.dim() != 2 or b.shape[1] != n or o.shape != a.shape or o.dtype != a.dtype or any(t.stride(1) != 1 for t in (a, b, o))
            or (ids is None and b.shape[0] != T) or (ids is not None and (ids.dtype != torch.int64 or ids.numel() != T or not ids.is_contiguous()))):
        raise TimeViperHipError(f"gated_mul: a {tuple(a.shape)} against b {tuple(b.shape)}")
    check(_capi.lib().tv_gated_mul_fwd(_p(a), _p(b), _p(ids), _p(o), T, n, a.stride(0), b.stride(0), o.stride(0), b.shape[0], int(act), _dt(a),
                                       _stream()), "tv_gated_mul_fwd")
    return o


def scatter_rows(src, rows, dst):
    """dst[rows] = src (rows int32 on the GPU, within dst)"""
    if src.is_cuda and _n.scatter_rows(src, rows, dst):
        return
    _gpu(src, rows, dst)
    _i32(rows, src.shape[0], "scatter_rows rows")
    if src.dtype != dst.dtype or src.shape[1] != dst.shape[1] or src.stride(1) != 1 or dst.stride(1) != 1:
        raise TimeViperHipError("scatter_rows: rows of one width and dtype")
    check(_capi.lib().tv_scatter_rows(_p(src), _p(rows), _p(dst), src.shape[0], src.shape[1], src.stride(0), dst.stride(0), _dt(src), _stream()),
          "tv_scatter_rows")


# ------------------------------------------------- linear attention with a constant decay per head
def lightning_attention(q, k, v, decay, state, cu_seqlens, slot, nheads, max_len, silu=True, out=None):
    """S_t = decay_h S_(t-1) + k_t v_t^T, o_t = S_t^T q_t for a ragged batch.  q, k (T, H * dk), v (T, H * dv): rows of a
    projection output (any row stride); decay (H) fp32; state (slots, H, dk, dv) fp32, advanced in place for the slots of this
    batch; cu_seqlens (B + 1) / slot (B) int32 on the GPU; max_len: the longest sequence's rows.  `silu`: q, k, v pass through SiLU here.  Returns (T, H * dv)."""
    _gpu(q, k, v, decay, state, cu_seqlens, slot)
    B = slot.numel()
    _i32(cu_seqlens, B + 1, "lightning_attention cu_seqlens")
    _i32(slot, B, "lightning_attention slot")
    T = q.shape[0]
    _, H, dk, dv = state.shape
    if H != nheads or q.shape != (T, H * dk) or k.shape != q.shape or v.shape != (T, H * dv):
        raise TimeViperHipError(f"lightning_attention: q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)}, state {tuple(state.shape)}")
    if state.dtype != torch.float32 or not state.is_contiguous() or decay.dtype != torch.float32 or k.dtype != q.dtype or v.dtype != q.dtype:
        raise TimeViperHipError("lightning_attention: fp32 contiguous state and decay; q, k, v of one dtype")
    if any(t.stride(1) != 1 for t in (q, k, v)) or not (1 <= max_len <= T) or (max_len == 1 and T != B):
        raise TimeViperHipError("lightning_attention: dense rows; max_len rows in the longest sequence")
    _vec(decay, H, "lightning_attention decay")
    o = torch.empty((T, H * dv), dtype=q.dtype, device=q.device) if out is None else out
    lib = _capi.lib()
    nbytes = int(lib.tv_lightning_workspace_bytes(B, int(max_len), H, dk, dv, _dt(q))) if max_len > 1 else 0
    ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes else None
    check(lib.tv_lightning_fwd(
        _p(q), _p(k), _p(v), _p(decay), _p(state), _p(o), _p(cu_seqlens), _p(slot), B, int(max_len), _p(ws), nbytes, H, dk, dv,
        q.stride(0), k.stride(0), v.stride(0), o.stride(0), int(bool(silu)), _dt(q), _stream()), "tv_lightning_fwd")
    return o


# ------------------------------------------------- attention without shape limits, latent attention
NO_WINDOW = 2 ** 31 - 1


def attention_generic(q, k, v, cu_seqlens, scale, causal=True, sink=None, start=None, slot=None, window=NO_WINDOW, keep_first=0, gate=None,
                      out=None):
    """q (T, Hq, dk) packed rows of B sequences (cu_seqlens (B + 1) int32); k (blocks, Lk, Hkv, dk), v (blocks, Lk, Hkv, dv): sequence b
    reads block slot[b] (default b).  Row i of a sequence sees keys [0, start[b] + i] when causal — with a window, the last `window` of
    them and the first `keep_first`.  gate (T, Hq, dv): the result times sigmoid(gate).  Returns (T, Hq, dv)."""
    _gpu(q, k, v, cu_seqlens, sink, start, slot, gate, out)
    T, Hq, dk = q.shape
    B = cu_seqlens.numel() - 1
    Hkv, dv = k.shape[2], v.shape[3]
    for t, n, what in ((cu_seqlens, B + 1, "cu_seqlens"), (start, B, "start"), (slot, B, "slot")):
        _i32(t, n, "attention_generic " + what)
    if k.dtype != q.dtype or v.dtype != q.dtype or any(t.stride(-1) != 1 for t in (q, k, v)) or k.shape[3] != dk or v.shape[:3] != k.shape[:3]:
        raise TimeViperHipError("attention_generic: q, k, v of one dtype with dense last dims and matching shapes")
    if sink is not None:
        if sink.dtype != torch.float32:
            raise TimeViperHipError("attention_generic: fp32 sinks")
        _vec(sink, Hq, "attention_generic sink")
    o = torch.empty((T, Hq, dv), dtype=q.dtype, device=q.device) if out is None else out
    for t in (o, gate):
        if t is not None and (t.shape != (T, Hq, dv) or t.dtype != q.dtype or t.stride(2) != 1):
            raise TimeViperHipError("attention_generic: gate and out (T, Hq, dv) of q's dtype with dense last dims")
    check(_capi.lib().tv_attn_generic_fwd(
        _p(q), _p(k), _p(v), _p(sink), _p(o), _p(cu_seqlens), _p(start), _p(slot), B, T, Hq, Hkv, dk, dv, q.stride(0), q.stride(1),
        k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(1), float(scale),
        int(bool(causal)), int(window), int(keep_first), _p(gate), 0 if gate is None else gate.stride(0),
        0 if gate is None else gate.stride(1), _dt(q), _stream()), "tv_attn_generic_fwd")
    return o


def _cache_views(cache, kv_heads, dim, vdim):
    """keys (slots, capacity, kv_heads, dim) and values (slots, capacity, kv_heads, vdim) of rows that hold both side by side"""
    slots, cap, W = cache.shape
    if W != kv_heads * (dim + vdim) or not cache.is_contiguous():
        raise TimeViperHipError(f"cache rows of {W} elements for {kv_heads} x ({dim} + {vdim})")
    k, v = cache.split([kv_heads * dim, kv_heads * vdim], dim=2)
    return k.unflatten(2, (kv_heads, dim)), v.unflatten(2, (kv_heads, vdim))


def attention_window(q, cache, plan, kv_heads, scale, window=NO_WINDOW, keep_first=0, gate=None, out=None):
    """Causal attention of a step's packed rows against a slot cache that already holds the step's own keys and values: q (T, H, dk), cache
    (slots, capacity, kv_heads * (dk + dv)), a row = all keys, then all values; the query at position p sees keys (p - window, p]
    and the first `keep_first` of its sequence.  gate (T, H, dv): the result times sigmoid(gate).  out (T, H, dv).  plan: the step's
    `cache.StepPlan`."""
    if q.is_cuda and (r := _n.attention_window(q, cache, plan.counts, plan.starts, plan.slots, kv_heads, scale, window, keep_first, gate, out,
                                                 plan.rows, plan.seq, plan.cu, plan.start, plan.slot)) is not None:
        return r
    T, H, dk = q.shape
    dv = cache.shape[2] // kv_heads - dk
    k, v = _cache_views(cache, kv_heads, dk, dv)
    _, cu, start, slot = _plan(plan, T, "attention_window")
    if max(plan.slots) >= cache.shape[0] or max(a + n for a, n in zip(plan.starts, plan.counts)) > cache.shape[1]:
        raise TimeViperHipError("attention_window: the cache does not hold the step's tokens")
    o = torch.empty((T, H, dv), dtype=q.dtype, device=q.device) if out is None else out
    rows8 = lambda t: t is None or (all(s % 4 == 0 for s in t.stride()[:2]) and t.data_ptr() % 8 == 0 and t.stride(2) == 1)
    if not (q.dtype == torch.bfloat16 and cache.dtype == q.dtype and _flash_rows(q) and _flash_rows(k[0]) and _flash_rows(v[0]) and rows8(gate)
            and rows8(o) and scale > 0):
        return attention_generic(q, k, v, cu, scale, start=start, slot=slot, window=window, keep_first=keep_first, gate=gate, out=o)
    _gpu(q, cache, gate, o)
    if H % kv_heads or any(t is not None and (t.shape != (T, H, dv) or t.dtype != q.dtype) for t in (gate, o)):
        raise TimeViperHipError("attention_window: gate and out (T, H, dv) of q's dtype")
    n = len(plan.counts)
    ints = lambda v: (ctypes.c_int * n)(*v)
    rows = [sum(plan.counts[:i]) for i in range(n)]
    check(_capi.lib().tv_flash_attn_window_packed_fwd(
        _p(q), _p(k), _p(v), _p(o), _p(gate), int(window), int(keep_first), dv, n, ints(rows), ints(plan.counts),
        ints([a + c for a, c in zip(plan.starts, plan.counts)]), ints(plan.slots), H, kv_heads, dk, q.stride(0), q.stride(1), k.stride(0), k.stride(1),
        k.stride(2), v.stride(0), v.stride(1), v.stride(2), o.stride(0), o.stride(1), 0 if gate is None else gate.stride(0),
        0 if gate is None else gate.stride(1), float(scale), _dt(q), _stream()), "tv_flash_attn_window_packed_fwd")
    return o


def attention_window_decode(q, cache, plan, kv_heads, scale, window=NO_WINDOW, keep_first=0, gate=None, fresh=None, out=None):
    """`attention_window` for a step of single tokens: q (B, H, dk), gate (B, H, dv).  fresh (B, kv_heads * (dk + dv)): the step's own cache
    rows, which are written here (without it they are in the cache already).  Key counts are read on the device.  Returns (B, H, dv)
    (`out`: where to)."""
    B, H, dk = q.shape
    dv = cache.shape[2] // kv_heads - dk
    k, v = _cache_views(cache, kv_heads, dk, dv)
    _, cu, start, slot = _plan(plan, B, "attention_window_decode")
    if not plan.decode or max(plan.slots) >= cache.shape[0] or H % kv_heads:
        raise TimeViperHipError("attention_window_decode: one token per sequence, each with a slot of the cache")
    _gpu(q, cache, gate, fresh, out, plan.keys)
    _i32(plan.keys, B, "attention_window_decode keys")
    if fresh is not None and (fresh.shape != (B, cache.shape[2]) or fresh.dtype != cache.dtype or fresh.stride(1) != 1):
        raise TimeViperHipError("attention_window_decode: new rows of the cache's width and dtype")
    dense = lambda t: t is None or (t.stride(2) == 1 and t.stride(1) == t.shape[2])
    ok16 = lambda t: t is None or (t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0)
    if (q.dtype == torch.bfloat16 and cache.dtype == q.dtype and dk % 8 == 0 and dv % 8 == 0 and max(dk, dv) <= 256 and dense(q) and dense(gate)
            and dense(out) and ok16(q) and ok16(fresh) and ok16(cache)):
        if any(t is not None and (t.shape != (B, H, dv) or t.dtype != q.dtype) for t in (gate, out)):
            raise TimeViperHipError("attention_window_decode: gate and out (B, H, dv) of q's dtype")
        o = torch.empty((B, H, dv), dtype=q.dtype, device=q.device) if out is None else out
        lib, cap = _capi.lib(), cache.shape[1]
        nbytes = int(lib.tv_attn_window_decode_workspace_bytes(B, H, kv_heads, dv, cap, int(window), int(keep_first)))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes else None
        check(lib.tv_attn_window_decode_fwd(
            _p(q), _p(cache), _p(fresh), _p(gate), _p(o), _p(plan.keys), _p(slot), B, H, kv_heads, dk, dv, cap, int(window), int(keep_first),
            q.stride(0), 0 if fresh is None else fresh.stride(0), 0 if gate is None else gate.stride(0), o.stride(0), float(scale), _p(ws), nbytes,
            _stream()), "tv_attn_window_decode_fwd")
        return o
    if fresh is not None:
        scatter_rows(fresh, plan.rows, cache.view(-1, cache.shape[2]))
    return attention_generic(q, k, v, cu, scale, start=start, slot=slot, window=window, keep_first=keep_first, gate=gate, out=out)


def _flash_rows(t: torch.Tensor) -> bool:
    """(rows, heads, dim) operands of tv_flash_attn_sink_fwd"""
    return t.shape[-1] % 8 == 0 and t.shape[-1] <= 128 and t.stride(-1) == 1 and all(s % 8 == 0 for s in t.stride()[:2]) \
        and t.data_ptr() % 16 == 0


def _flash_sink(q, k, v, counts, starts, scale, sink):
    T, Hq, D = q.shape
    Hkv, Dv = k.shape[1], v.shape[2]
    _gpu(q, k, v, sink)
    o = torch.empty((T, Hq, Dv), dtype=q.dtype, device=q.device)
    lib, at, kt = _capi.lib(), 0, 0
    for n, a in zip(counts, starts):
        qb, kb, vb, ob = q[at:at + n], k[kt:kt + a + n], v[kt:kt + a + n], o[at:at + n]
        check(lib.tv_flash_attn_sink_fwd(
            _p(qb), _p(kb), _p(vb), _p(ob), _p(sink), Dv, 1, n, a + n, Hq, Hkv, D, 0, q.stride(0), q.stride(1), 0, k.stride(0), k.stride(1),
            0, v.stride(0), v.stride(1), 0, o.stride(0), o.stride(1), float(scale), _dt(q), _stream()), "tv_flash_attn_sink_fwd")
        at, kt = at + n, kt + a + n
    return o


def attention_sink(q, k, v, cu_q, cu_k, start, counts, starts, scale, sink):
    """Causal attention over a ragged batch with a sink logit per head.  q (T, H, dk): sequence b owns rows [cu_q[b], cu_q[b + 1]);
    k (Tk, H, dk), v (Tk, H, dv): rows [cu_k[b], cu_k[b + 1]), start[b] = the keys in front of the sequence's first query row
    (int32 tensors on the GPU; `counts` / `starts`: the same per sequence on the host).  Returns (T, H, dv)."""
    if q.dtype == torch.bfloat16 and all(_flash_rows(t) for t in (q, k, v)):
        return _flash_sink(q, k, v, counts, starts, scale, sink)
    blocks = lambda t: t.as_strided((t.shape[0], 1) + t.shape[1:], (t.stride(0),) + t.stride())      # a "block" per row: slot = first row
    return attention_generic(q, blocks(k), blocks(v), cu_q, scale, sink=sink, start=start, slot=cu_k[:-1])


def _latent_args(t, w, nheads, what):
    if t.dtype != w.dtype or t.stride(1) != 1 or w.stride(1) != 1 or t.shape[1] % nheads or w.shape[0] % nheads:
        raise TimeViperHipError(f"{what}: operands of one dtype with dense rows, heads contiguous")


def latent_query(q, w_uk, nheads):
    """(B, H * dim), W_uk (H * dim, rank) -> (B, H, rank): the query against the latents themselves."""
    _gpu(q, w_uk)
    _latent_args(q, w_uk, nheads, "latent_query")
    B, rank, dim = q.shape[0], w_uk.shape[1], w_uk.shape[0] // nheads
    if q.shape[1] != nheads * dim:
        raise TimeViperHipError("latent_query: q and W_uk disagree about the head size")
    y = torch.empty((B, nheads, rank), dtype=q.dtype, device=q.device)
    check(_capi.lib().tv_latent_query_fwd(_p(q), _p(w_uk), _p(y), B, nheads, dim, rank, q.stride(0), w_uk.stride(0), y.stride(0), _dt(q),
                                          _stream()), "tv_latent_query_fwd")
    return y


def latent_value(y, w_uv, nheads):
    """(B, H, rank), W_uv (H * vdim, rank) -> (B, H * vdim)."""
    _gpu(y, w_uv)
    B, H, rank = y.shape
    vdim = w_uv.shape[0] // nheads
    if H != nheads or w_uv.shape != (H * vdim, rank) or not y.is_contiguous() or w_uv.stride(1) != 1 or y.dtype != w_uv.dtype:
        raise TimeViperHipError("latent_value: y (B, H, rank) contiguous, W_uv (H * vdim, rank)")
    o = torch.empty((B, H * vdim), dtype=y.dtype, device=y.device)
    check(_capi.lib().tv_latent_value_fwd(_p(y), _p(w_uv), _p(o), B, H, vdim, rank, y.stride(0), w_uv.stride(0), o.stride(0), _dt(y),
                                          _stream()), "tv_latent_value_fwd")
    return o


def latent_decode(q, w_uk, w_uv, latents, keys, slot, nheads, scale, sink, new=None):
    """One token per sequence: q (B, H * dim) against the first keys[b] (int32, on the GPU) rows of latents[slot[b]] (slots, capacity,
    rank) -> (B, H * vdim), what attention over the expanded keys W_uk c and values W_uv c gives.
    `new=(c, norm_weight, eps, rows)`: the step's own down projections (B, rank); their normed rows go to the cache rows `rows` (of
    the (slots * capacity, rank) view) first."""
    _gpu(q, w_uk, w_uv, latents, keys, slot, sink)
    B, R = q.shape[0], latents.shape[2]
    _latent_args(q, w_uk, nheads, "latent_decode")
    dim, vdim = w_uk.shape[0] // nheads, w_uv.shape[0] // nheads
    _i32(keys, B, "latent_decode keys")
    _i32(slot, B, "latent_decode slot")
    if (q.shape[1] != nheads * dim or w_uk.shape[1] != R or w_uv.shape != (nheads * vdim, R) or latents.dtype != q.dtype
            or w_uv.dtype != q.dtype or not latents.is_contiguous()):
        raise TimeViperHipError("latent_decode: q, W_uk, W_uv and the latents disagree")
    if new is not None:
        c, cn, _, rows = new
        _gpu(c, cn, rows)
        _i32(rows, B, "latent_decode rows")
        _vec(cn, R, "latent_decode norm weight")
        if c.shape != (B, R) or c.dtype != q.dtype or cn.dtype != q.dtype or c.stride(1) != 1:
            raise TimeViperHipError("latent_decode: new latents (B, rank) of the model's dtype")
    if (q.dtype == torch.bfloat16 and R % 8 == 0 and R <= 512 and w_uk.is_contiguous() and w_uv.is_contiguous()
            and all(t.data_ptr() % 16 == 0 for t in (w_uk, w_uv, latents))):
        _vec(sink, nheads, "latent_decode sink")
        c, cn, eps, rows = new if new is not None else (None, None, 0.0, None)
        o = torch.empty((B, nheads * vdim), dtype=q.dtype, device=q.device)
        lib = _capi.lib()
        nbytes = int(lib.tv_latent_decode_workspace_bytes(B, nheads, R, latents.shape[1]))
        ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device)
        check(lib.tv_latent_decode_fwd(
            _p(q), _p(w_uk), _p(w_uv), _p(latents), _p(c), _p(cn), float(eps), _p(rows), _p(keys), _p(slot), _p(sink), _p(o), B, nheads,
            dim, vdim, R, latents.shape[1], q.stride(0), 0 if c is None else c.stride(0), o.stride(0), float(scale), _p(ws), nbytes,
            _stream()), "tv_latent_decode_fwd")
        return o
    if new is not None:
        rms_norm_ex(new[0], new[1], new[2], y2=latents.view(-1, R), y2_rows=new[3], need_y=False)
    ql = latent_query(q, w_uk, nheads)
    kv = latents.unsqueeze(2)                                   # one shared key / value head of `rank` dimensions
    cu = torch.arange(B + 1, dtype=torch.int32, device=q.device)
    y = attention_generic(ql, kv, kv, cu, scale, sink=sink, start=keys - 1, slot=slot)
    return latent_value(y, w_uv, nheads)


# ------------------------------------------------- decode-step linear layers of post-norm models
GEMV_POSTNORM, GEMV_NORMGATE = 4, 5


def gemv_post_takes(rows: int, width: int, dtype) -> bool:
    """Shapes of tv_gemv_post_fwd with a norm prologue: 1..4 bf16 rows of up to 8 192 elements."""
    return dtype == torch.bfloat16 and 1 <= rows <= 4 and width % 8 == 0 and width <= 8192 and rows * width * 2 <= 128 * 1024


def gemv_post(x, weight, prologue=GEMV_NONE, residual=None, norm_weight=None, eps=0.0, weight_offset=0.0, mult=1.0, gate=None,
              out_dtype=torch.bfloat16):
    """y = f(x) @ weight.T for 1..4 bf16 rows.  GEMV_NONE: f(x) = x.  GEMV_POSTNORM: the norm of a sublayer's output x, the residual
    add x' = residual + mult * rms(x) * (weight_offset + norm_weight) in fp32, f = x' in bf16; returns (y, x', bf16 x').
    GEMV_NORMGATE: f = rms(x) * norm_weight * sigmoid(gate)."""
    _gpu(x, weight, residual, norm_weight, gate)
    M, Kd = x.shape
    N = weight.shape[0]
    if x.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16 or weight.shape[1] != Kd or x.stride(1) != 1 or weight.stride(1) != 1:
        raise TimeViperHipError(f"gemv_post: bf16 rows x {tuple(x.shape)} against weight {tuple(weight.shape)}")
    y = torch.empty((M, N), dtype=out_dtype, device=x.device)
    xs = hs = None
    if prologue == GEMV_POSTNORM:
        if residual is None or residual.dtype != torch.float32 or residual.shape != x.shape or not residual.is_contiguous():
            raise TimeViperHipError("gemv_post: a dense fp32 residual of x's shape")
        xs, hs = torch.empty_like(residual), torch.empty((M, Kd), dtype=x.dtype, device=x.device)
    if gate is not None and (gate.shape != x.shape or gate.dtype != x.dtype or gate.stride(1) != 1):
        raise TimeViperHipError("gemv_post: gate must have x's shape and dtype")
    if norm_weight is not None:
        _vec(norm_weight, Kd, "gemv_post norm weight")
    check(_capi.lib().tv_gemv_post_fwd(
        _p(x), _p(weight), _p(y), _DT[out_dtype], M, N, Kd, x.stride(0), weight.stride(0), N, int(prologue), _p(residual), _p(xs), _p(hs),
        _p(norm_weight), 0 if norm_weight is None else _dt(norm_weight), float(weight_offset), float(mult), float(eps), _p(gate),
        0 if gate is None else gate.stride(0), _stream()), "tv_gemv_post_fwd")
    return (y, xs, hs) if prologue == GEMV_POSTNORM else y


def gemv_rows_take(rows: int, width: int, dtype) -> bool:
    """Shapes of gemv_pair, gemv_add and gemv_glu: 1..4 bf16 rows that fit the LDS."""
    return dtype == torch.bfloat16 and 1 <= rows <= 4 and width % 8 == 0 and rows * width * 2 <= 128 * 1024


def _gemv_rows(what, weight, *rows):
    if weight.dtype != torch.bfloat16 or weight.dim() != 2 or weight.stride(1) != 1 or any(
            t.dtype != torch.bfloat16 or t.shape != rows[0].shape or t.shape[1] != weight.shape[1] or t.stride(1) != 1 for t in rows):
        raise TimeViperHipError(f"{what}: bf16 rows {tuple(rows[0].shape)} against weight {tuple(weight.shape)}")


def _bf16_bias(t, n, what):
    if t is not None:
        _vec(t, n, what)
        if t.dtype != torch.bfloat16:
            raise TimeViperHipError(f"{what}: bf16")


def gemv_pair(x, x2, weight, n1, bias=None, act_out=None, many=False):
    """Both input products of a parallel layer for 1..4 bf16 rows, one launch: y = x @ weight[:n1].T (returned) and, when weight has more
    rows (gate | up), act_out = gelu_tanh(x2 @ gate.T + b) * (x2 @ up.T + b), bias = their biases."""
    _gpu(x, x2, weight, bias, act_out)
    M, D = x.shape
    ff = (weight.shape[0] - n1) // 2
    _gemv_rows("gemv_pair", weight, x, *((x2,) if ff else ()))
    if weight.shape[0] != n1 + 2 * ff or n1 < 1 or (ff and (bias is None or act_out is None or act_out.shape != (M, ff) or act_out.dtype != x.dtype
                                                          or act_out.stride(1) != 1)):
        raise TimeViperHipError(f"gemv_pair: weight rows {n1} + 2 x {ff}, biases and an (M, {ff}) output for the second part")
    if ff:
        _bf16_bias(bias, 2 * ff, "gemv_pair bias")
    y = torch.empty((M, n1), dtype=x.dtype, device=x.device)
    lib = _capi.lib()
    fn, what = (lib.tv_gemv_pair_fwd, "tv_gemv_pair_fwd") if not many else (lib.tv_gemm_rows_pair_fwd, "tv_gemm_rows_pair_fwd")
    check(fn(_p(x), _p(x2) if ff else None, _p(weight), _p(bias), _p(y), _p(act_out) if ff else None, M, int(n1), ff, D,
             x.stride(0), x2.stride(0) if ff else 0, weight.stride(0), n1, act_out.stride(0) if ff else 0, _stream()), what)
    return y


def rows_pair(x, x2, weight, n1, bias=None, act_out=None):
    """gemv_pair for 2..32 rows (`rows_take`)"""
    return gemv_pair(x, x2, weight, n1, bias, act_out, many=True)


def gemv_add(x, weight, residual, bias=None, many=False):
    """(residual + x @ weight.T + bias in fp32, its bf16 rounding) for 1..4 bf16 rows; residual (M, N) fp32"""
    _gpu(x, weight, bias, residual)
    _gemv_rows("gemv_add", weight, x)
    M, N = x.shape[0], weight.shape[0]
    _bf16_bias(bias, N, "gemv_add bias")
    if residual.dtype != torch.float32 or residual.shape != (M, N) or not residual.is_contiguous():
        raise TimeViperHipError("gemv_add: a dense fp32 residual (M, N)")
    xo, h = torch.empty_like(residual), torch.empty((M, N), dtype=x.dtype, device=x.device)
    lib = _capi.lib()
    fn, what = (lib.tv_gemv_add_fwd, "tv_gemv_add_fwd") if not many else (lib.tv_gemm_rows_add_fwd, "tv_gemm_rows_add_fwd")
    check(fn(_p(x), _p(weight), _p(bias), _p(residual), _p(xo), _p(h), M, N, x.shape[1], x.stride(0), weight.stride(0), _stream()), what)
    return xo, h


def rows_add(x, weight, residual, bias=None):
    """gemv_add for 2..32 rows (`rows_take`)"""
    return gemv_add(x, weight, residual, bias, many=True)


def gemv_glu(z, u, weight, ids=None):
    """(gelu_tanh(z) * u) @ weight.T for 1..4 bf16 rows; `ids` (int64): row m meets u[ids[m]]"""
    _gpu(z, u, weight, ids)
    _gemv_rows("gemv_glu", weight, z)
    M, N = z.shape[0], weight.shape[0]
    if (u.dtype != z.dtype or u.stride(1) != 1 or u.shape[1] != z.shape[1] or (ids is None and u.shape[0] != M)
            or (ids is not None and (ids.dtype != torch.int64 or ids.numel() != M or not ids.is_contiguous()))):
        raise TimeViperHipError("gemv_glu: u rows of z's width, one per row or by int64 ids")
    y = torch.empty((M, N), dtype=z.dtype, device=z.device)
    check(_capi.lib().tv_gemv_glu_fwd(_p(z), _p(u), _p(ids), u.shape[0], _p(weight), _p(y), M, N, z.shape[1], z.stride(0), u.stride(0), weight.stride(0),
                                      N, _stream()), "tv_gemv_glu_fwd")
    return y


def rows_glu_takes(x, weight, u) -> bool:
    """Operands tv_gemm_rows_glu_fwd reads: 2..32 rows as `rows_take`, at most 8 outputs a compute unit, rows of u of one width"""
    return (x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.stride(0) < (1 << 24) and x.data_ptr() % 16 == 0 and rows_take(x, weight)
            and weight.shape[0] <= 8 * CUS and u.dtype == x.dtype and u.dim() == 2 and u.stride(1) == 1 and u.shape[1] == weight.shape[0])


def rows_glu(x, weight, u, ids=None):
    """gelu_tanh(x @ weight.T) * u for 2..32 bf16 rows, the product rounded in front of the activation; `ids` (int64): row m meets u[ids[m]]"""
    _gpu(x, weight, u, ids)
    M, (N, Kd) = x.shape[0], weight.shape
    if (not rows_glu_takes(x, weight, u) or x.shape[1] != Kd or (ids is None and u.shape[0] != M)
            or (ids is not None and (ids.dtype != torch.int64 or ids.numel() != M or not ids.is_contiguous()))):
        raise TimeViperHipError(f"rows_glu: rows {tuple(x.shape)} against {tuple(weight.shape)}, u {tuple(u.shape)}, one per row or by int64 ids")
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    check(_capi.lib().tv_gemm_rows_glu_fwd(_p(x), _p(weight), _p(u), _p(ids), u.shape[0], _p(y), M, N, Kd, x.stride(0), weight.stride(0), u.stride(0), N,
                                           _stream()), "tv_gemm_rows_glu_fwd")
    return y


# ------------------------------------------------- mixture of experts
MOE_NONE, MOE_RELU2 = 0, 1


def moe_router(x, weight, correction, top):
    """softmax router: (ids (T, top) int32, weights (T, top) fp32) of the `top` outputs with the largest softmax + correction; the
    weights are the softmax values."""
    _gpu(x, weight, correction)
    T, D = x.shape
    E = weight.shape[0]
    if weight.shape[1] != D or not weight.is_contiguous() or x.stride(1) != 1:
        raise TimeViperHipError("moe_router: x (T, D), weight (outputs, D)")
    if correction is not None:
        _vec(correction, E, "moe_router correction")
        if correction.dtype != weight.dtype:
            raise TimeViperHipError("moe_router: correction of the weight's dtype")
    ids = torch.empty((T, top), dtype=torch.int32, device=x.device)
    w = torch.empty((T, top), dtype=torch.float32, device=x.device)
    check(_capi.lib().tv_moe_router_fwd(_p(x), _p(weight), _p(correction), _p(ids), _p(w), T, D, E, top, x.stride(0), _dt(x), _dt(weight),
                                        _stream()), "tv_moe_router_fwd")
    return ids, w


def moe_plan(ids, experts):
    """The choices (T, top) sorted by expert: (offsets (experts + 1), row_token (T * top), pos (T, top)) int32; pos -1: id >= experts
    (an identity expert, no row)."""
    _gpu(ids)
    T, top = ids.shape
    _i32(ids, T * top, "moe_plan ids")
    dev = ids.device
    counts = torch.empty(experts, dtype=torch.int32, device=dev)
    offsets = torch.empty(experts + 1, dtype=torch.int32, device=dev)
    row_token = torch.empty(T * top, dtype=torch.int32, device=dev)
    pos = torch.empty((T, top), dtype=torch.int32, device=dev)
    check(_capi.lib().tv_moe_plan(_p(ids), _p(counts), _p(offsets), _p(row_token), _p(pos), T * top, experts, top, _stream()), "tv_moe_plan")
    return offsets, row_token, pos


def moe_gemm(a, w, offsets, max_rows, row_token=None, act=MOE_NONE):
    """C (max_rows, N): rows [offsets[e], offsets[e + 1]) = act(a[row_token] @ w[e].T); w (experts, N, K)."""
    _gpu(a, w, offsets, row_token)
    E, N, Kd = w.shape
    _i32(offsets, E + 1, "moe_gemm offsets")
    _i32(row_token, max_rows, "moe_gemm row_token")
    if a.shape[1] != Kd or a.dtype != w.dtype or a.stride(1) != 1 or not w.is_contiguous() or (row_token is None and a.shape[0] < max_rows):
        raise TimeViperHipError(f"moe_gemm: a {tuple(a.shape)} against w {tuple(w.shape)}")
    c = torch.empty((max_rows, N), dtype=a.dtype, device=a.device)
    check(_capi.lib().tv_moe_gemm_fwd(_p(a), _p(w), _p(c), _p(offsets), _p(row_token), a.shape[0], max_rows, E, N, Kd, a.stride(0), c.stride(0), int(act),
                                      _dt(a), _stream()), "tv_moe_gemm_fwd")
    return c


def moe_decode_takes(tokens: int, n_out: int, top: int, width: int, ff: int, dtype) -> bool:
    """Shapes of tv_moe_decode_fwd."""
    return (dtype == torch.bfloat16 and tokens <= 4 and n_out <= 256 and top <= 32 and width % 8 == 0 and width <= 8192 and ff % 8 == 0
            and top * ff * 2 <= 128 * 1024)


def moe_decode(logits, correction, h, x, up, down, top):
    """Mixture of experts for a few single tokens: router logits (T, outputs) fp32, h (T, D) bf16 and the fp32 rows x it was rounded from,
    up (E, ff, D), down (E, D, ff).  Returns (sum of the chosen experts' outputs (T, D) bf16, ids (T, top) int32)."""
    _gpu(logits, correction, h, x, up, down)
    T, D = h.shape
    E, ff, _ = up.shape
    n_out = logits.shape[1]
    if (logits.shape != (T, n_out) or logits.dtype != torch.float32 or not logits.is_contiguous() or up.shape != (E, ff, D)
            or down.shape != (E, D, ff) or x.shape != h.shape or x.dtype != torch.float32 or any(t.dtype != torch.bfloat16 for t in (h, up, down, correction))
            or not all(t.is_contiguous() for t in (h, x, up, down))):
        raise TimeViperHipError("moe_decode: dense fp32 logits and x, dense bf16 h, up and down of matching sizes")
    _vec(correction, n_out, "moe_decode correction")
    dev = h.device
    ids = torch.empty((T, top), dtype=torch.int32, device=dev)
    wts = torch.empty((T, top), dtype=torch.float32, device=dev)
    u = torch.empty((T * top, ff), dtype=h.dtype, device=dev)
    y = torch.empty((T, D), dtype=h.dtype, device=dev)
    check(_capi.lib().tv_moe_decode_fwd(_p(logits), _p(correction), _p(h), _p(x), _p(up), _p(down), _p(ids), _p(wts), _p(u), _p(y), T, E, n_out, top,
                                        D, ff, _stream()), "tv_moe_decode_fwd")
    return y, ids
