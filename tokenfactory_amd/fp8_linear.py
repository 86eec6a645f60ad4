"""Block-FP8 linear layers on the gfx950 kernels.

``block_fp8_linear`` is the native counterpart of the reference's
``triton_block_fp8_linear(x, weight, weight_scale_inv, bias, block_h, block_w)``
(``qwen3_8/fp8_triton.py:107-183``): dynamic per-tensor quantisation of the
activations to e4m3 (``tf_fp8_act_quant``) followed by the block-scaled FP8
GEMM (``tf_fp8_block_gemm``), bf16 in and out.

``Fp8Linear`` mirrors ``Qwen3_8FP8Linear`` (``qwen3_8/fp8_linear.py:12-212``)
for a float8_e4m3fn weight: the same parameter and buffer names and shapes
(``weight`` ``[out, in]``, ``weight_scale_inv`` ``[ceil(out / block_h),
ceil(in / block_w)]``), ``dequantize_weight`` with the reference's
expand-and-multiply semantics, and a forward that always runs the native GEMM.
There is no non-native path: without the library every call raises.
"""
from __future__ import annotations

import contextlib
import math
from typing import Optional, Sequence

import torch
import torch.nn as nn

from . import _native

FP8_MAX = 448.0


def _ptr(t: Optional[torch.Tensor]) -> int:
    return 0 if t is None else t.data_ptr()


def _stream_ptr(stream, device) -> int:
    return stream.cuda_stream if stream is not None else _native.current_stream(device)


def on_stream(stream):
    """Context that makes ``stream`` current (a no-op for None), so that the
    temporaries a call allocates and the torch ops it runs are ordered on the
    stream its kernels run on, and the caching allocator reuses their memory
    only after that stream is done with it."""
    return torch.cuda.stream(stream) if stream is not None else contextlib.nullcontext()


K_SLICE = 128   # the GEMM's K granularity (one weight-scale block)


def _padded_k(k: int) -> int:
    return -(-k // K_SLICE) * K_SLICE


def _pad_cols(t: torch.Tensor, cols: int) -> torch.Tensor:
    """``t`` with zero columns appended up to ``cols`` (zero e4m3 products add
    nothing to any sum)."""
    if t.shape[1] == cols:
        return t
    out = torch.zeros((t.shape[0], cols), dtype=torch.uint8, device=t.device)
    out[:, : t.shape[1]] = t.view(torch.uint8)
    return out.view(t.dtype)


def _check_amax(amax: Optional[torch.Tensor], x2d: torch.Tensor, limit: int) -> None:
    if amax is not None and (amax.dtype != torch.int32 or not 1 <= amax.numel() <= limit
                             or amax.device != x2d.device or not amax.is_contiguous()):
        raise ValueError(f"the amax of x must be a contiguous int32 tensor on x's device with "
                         f"1 to {limit} elements")


def quantize_activations(x2d: torch.Tensor, stream=None, padded_cols: Optional[int] = None,
                         amax: Optional[torch.Tensor] = None):
    """Dynamic per-tensor e4m3 quantisation of a bf16 ``[rows, cols]`` matrix
    (``fp8_triton.py:127-130``). Returns ``(xq, x_scale)``: float8_e4m3fn rows
    and a 1-element fp32 tensor holding ``bf16(max(amax|x|, 1e-12) / 448)``.
    With ``padded_cols`` the rows of ``xq`` are zero-extended to that width.
    ``amax``: the max of ``|x|`` already computed by x's producer (a 1-element
    int32 device tensor holding the bf16 bit pattern, as the attention kernels'
    ``out_amax`` leaves it); the result is the same, with one launch
    (``tf_fp8_act_quant_amax``) instead of two."""
    if x2d.dtype != torch.bfloat16 or x2d.dim() != 2 or not x2d.is_cuda:
        raise ValueError("quantize_activations: x must be a 2-D bf16 CUDA tensor")
    if x2d.stride(1) != 1:
        raise ValueError("quantize_activations: x rows must be contiguous")
    rows, cols = x2d.shape
    width = cols if padded_cols is None else padded_cols
    if width < cols:
        raise ValueError("quantize_activations: padded_cols < cols")
    with on_stream(stream):
        xq = torch.empty((rows, width), dtype=torch.float8_e4m3fn, device=x2d.device)
        if width > cols:
            xq.view(torch.uint8)[:, cols:].zero_()
        scale = torch.empty((1,), dtype=torch.float32, device=x2d.device)
        if amax is not None:
            _check_amax(amax, x2d, 1)
            _native.call("tf_fp8_act_quant_amax", _ptr(x2d), _native.TF_DTYPE_BF16, rows, cols,
                         x2d.stride(0), _ptr(xq), xq.stride(0), _ptr(scale), _ptr(amax),
                         _stream_ptr(stream, x2d.device))
            return xq, scale
        ws = torch.empty((_native.TF_FP8_QUANT_WORKSPACE_BYTES,), dtype=torch.uint8,
                         device=x2d.device)
        _native.call("tf_fp8_act_quant", _ptr(x2d), _native.TF_DTYPE_BF16, rows, cols,
                     x2d.stride(0), _ptr(xq), xq.stride(0), _ptr(scale), _ptr(ws), ws.numel(),
                     _stream_ptr(stream, x2d.device))
    return xq, scale


def block_fp8_gemm(xq: torch.Tensor, x_scale: torch.Tensor, weight: torch.Tensor,
                   weight_scale_inv: Optional[torch.Tensor], bias: Optional[torch.Tensor],
                   block_h: int = 128, block_w: int = 128, out: Optional[torch.Tensor] = None,
                   stream=None) -> torch.Tensor:
    """``bf16(sum_kb (xq w^T)[:, kb] * x_scale * weight_scale_inv[n // block_h,
    kb // block_w] + bias)`` (``fp8_triton.py:17-98``), fp32 accumulation.

    ``xq`` may carry zero columns beyond ``weight``'s width (up to the next
    multiple of 128); a width that is not a multiple of 128 is zero-padded
    here, since the kernel consumes K in 128-wide slices."""
    if xq.dtype != torch.float8_e4m3fn or weight.dtype != torch.float8_e4m3fn:
        raise ValueError("block_fp8_gemm: xq and weight must be float8_e4m3fn")
    if xq.dim() != 2 or weight.dim() != 2:
        raise ValueError(f"block_fp8_gemm: shapes {tuple(xq.shape)} x {tuple(weight.shape)}^T")
    k = weight.shape[1]
    kp = _padded_k(k)
    if xq.shape[1] not in (k, kp):
        raise ValueError(f"block_fp8_gemm: shapes {tuple(xq.shape)} x {tuple(weight.shape)}^T")
    if xq.stride(1) != 1 or weight.stride(1) != 1:
        raise ValueError("block_fp8_gemm: xq / weight rows must be contiguous")
    m = xq.shape[0]
    n = weight.shape[0]
    if weight_scale_inv is not None:
        if weight_scale_inv.dtype != torch.float32:
            raise ValueError("block_fp8_gemm: weight_scale_inv must be float32")
        need = (math.ceil(n / block_h), math.ceil(k / block_w))
        if tuple(weight_scale_inv.shape) != need:
            raise ValueError(f"block_fp8_gemm: weight_scale_inv {tuple(weight_scale_inv.shape)}, "
                             f"expected {need}")
    if bias is not None and (bias.dtype != torch.bfloat16 or bias.shape != (n,)
                             or bias.stride(0) != 1):
        raise ValueError("block_fp8_gemm: bias must be a contiguous bf16 [out_features]")
    if x_scale.dtype != torch.float32 or x_scale.numel() != 1:
        raise ValueError("block_fp8_gemm: x_scale must be a 1-element float32 tensor")
    if out is not None and (out.dtype != torch.bfloat16 or tuple(out.shape) != (m, n)
                            or out.stride(1) != 1):
        raise ValueError("block_fp8_gemm: out must be bf16 [m, n] with contiguous rows")
    # split-K scratch for small m (0 bytes when the call does not split)
    nbytes = _native.load().tf_fp8_block_gemm_workspace_bytes(m, n, kp) if m > 0 else 0
    if nbytes < 0:
        raise ValueError("block_fp8_gemm: bad shape")
    with on_stream(stream):
        if out is None:
            out = torch.empty((m, n), dtype=torch.bfloat16, device=xq.device)
        ws = weight_scale_inv
        if kp != k:
            xq, weight = _pad_cols(xq, kp), _pad_cols(weight, kp)
            if ws is None:        # one all-ones block over the true K (fp8_triton.py:132-135)
                block_w = kp
        scratch = torch.empty((nbytes,), dtype=torch.uint8, device=xq.device) if nbytes else None
        _native.call("tf_fp8_block_gemm", _ptr(xq), xq.stride(0), _ptr(x_scale),
                     _ptr(weight), weight.stride(0), _ptr(ws),
                     0 if ws is None else ws.stride(0), 0 if ws is None else ws.stride(1),
                     block_h, block_w, _ptr(bias), m, n, kp, _ptr(out), out.stride(0),
                     _ptr(scratch), nbytes, _stream_ptr(stream, xq.device))
    return out


def _takes(x2d: torch.Tensor) -> bool:
    """Whether x is what ``tf_fp8_linears`` takes (else: the calls step by step,
    which pad a K that is not a multiple of 128, or say what is wrong)."""
    return x2d.is_cuda and x2d.dtype == torch.bfloat16 and x2d.shape[1] % K_SLICE == 0


def _shared(x2d: torch.Tensor, w: torch.Tensor, scale: Optional[torch.Tensor],
            bias: Optional[torch.Tensor], block_h: int, block_w: int) -> bool:
    """Whether one weight of block size (block_h, block_w) is what
    ``tf_fp8_linears`` takes with x."""
    dev = x2d.device
    if (w.dtype != torch.float8_e4m3fn or w.dim() != 2 or w.device != dev
            or not w.is_contiguous() or scale is None or scale.dtype != torch.float32
            or scale.device != dev):
        return False
    n, k = w.shape
    return (k == x2d.shape[1] and scale.shape == (-(-n // block_h), -(-k // block_w))
            and (bias is None or (bias.dtype == torch.bfloat16 and bias.shape == (n,)
                                  and bias.device == dev and bias.is_contiguous())))


def _linears(x2d: torch.Tensor, weights, block_h: int, block_w: int,
             amax: Optional[torch.Tensor] = None, stream=None):
    """``[x2d w^T + bias]`` for (weight, scales, bias) triples that pass
    ``_takes`` and ``_shared``, in one ``tf_fp8_linears`` call: one entry and
    one workspace for the quantisation and the GEMM, since at decode sizes the
    host's calls and allocations take longer than the kernels (full-attention
    layer, 16 decodes: host 150 -> 109 us a call, kernels 97)."""
    rows, k = x2d.shape
    dev = x2d.device
    n = len(weights)
    mats = (_native.Fp8Mat * n)()
    lib = _native.load()
    with on_stream(stream):
        outs = [torch.empty((rows, w.shape[0]), dtype=torch.bfloat16, device=dev)
                for w, _, _ in weights]
        for i, (w, scale, bias) in enumerate(weights):
            cols = w.shape[0]
            mats[i] = (w.data_ptr(), k, scale.data_ptr(), scale.stride(0), scale.stride(1),
                       _ptr(bias), cols, outs[i].data_ptr(), cols)
        if rows:
            nbytes = lib.tf_fp8_linears_workspace_bytes(rows, mats, n, k)
            ws = torch.empty((max(nbytes, 0),), dtype=torch.uint8, device=dev)
            _native.call("tf_fp8_linears", x2d.data_ptr(), x2d.stride(0), _ptr(amax),
                         0 if amax is None else amax.numel(), mats, n, block_h, block_w, rows, k,
                         ws.data_ptr(), nbytes, _stream_ptr(stream, dev))
    return outs


def block_fp8_linear(x: torch.Tensor, weight: torch.Tensor,
                     weight_scale_inv: Optional[torch.Tensor], bias: Optional[torch.Tensor],
                     block_h: int = 128, block_w: int = 128, stream=None,
                     x_amax: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Native ``triton_block_fp8_linear`` (``fp8_triton.py:107-183``): x ``[..., in]``
    bf16, weight float8_e4m3fn ``[out, in]`` -> bf16 ``[..., out]``. ``x_amax``:
    max ``|x|`` from x's producer, see ``quantize_activations``."""
    in_features = weight.shape[1]
    if x.shape[-1] != in_features:
        raise ValueError(f"block_fp8_linear: x [..., {x.shape[-1]}] vs weight in={in_features}")
    x2d = x.reshape(-1, in_features)
    if x2d.stride(1) != 1:
        x2d = x2d.contiguous()
    if x2d.shape[0] and _takes(x2d) and _shared(x2d, weight, weight_scale_inv, bias, block_h,
                                                block_w):
        _check_amax(x_amax, x2d, 1)
        out, = _linears(x2d, ((weight, weight_scale_inv, bias),), block_h, block_w, x_amax, stream)
        return out.reshape(*x.shape[:-1], weight.shape[0])
    xq, scale = quantize_activations(x2d, stream, padded_cols=_padded_k(in_features),
                                     amax=x_amax)
    out = block_fp8_gemm(xq, scale, weight, weight_scale_inv, bias, block_h, block_w,
                         stream=stream)
    return out.reshape(*x.shape[:-1], weight.shape[0])


def _plain(linear, kind) -> bool:
    """Whether calling ``linear`` runs ``kind.forward`` on plain tensors and nothing
    else (no subclass of the module or of its weight, replaced forward or hook)."""
    return (type(linear) is kind and "forward" not in linear.__dict__
            and type(linear._parameters.get("weight")) is nn.Parameter
            and not (linear._forward_hooks or linear._forward_pre_hooks
                     or linear._backward_hooks or linear._backward_pre_hooks
                     or nn.modules.module._has_any_global_hook()))


# Elements of x up to which the gate projections share a launch.  Above, the
# library's two products and a pass for max |x| are faster: its kernel re-reads x for
# each 32 columns of either weight, from memory once x outgrows the caches
# (hidden 5120, 48 + 48 columns, us shared / two products + pass: 4000 rows 37 / 51,
# 5000 53 / 53, 8000 73 / 56, 16000 142 / 91; hidden 8192, 64 + 64: 3000 62 / 69,
# 5000 93 / 63; hidden 2048, 32 + 32: 12000 32 / 51).
NARROW_MAX_ELEMS = 24 << 20


def _narrow_pair(x: torch.Tensor, first: nn.Module, second: nn.Module):
    """The weights of the pair if ``tf_narrow_linear2`` takes it, else None.  (The
    modules may be anything that can be called: nothing of them is read before they
    are known to be plain.)"""
    if not (_plain(first, nn.Linear) and _plain(second, nn.Linear)):
        return None
    pair = w0, w1 = first.weight, second.weight
    n, k = w0.shape
    if torch.is_grad_enabled() and (x.requires_grad or w0.requires_grad or w1.requires_grad):
        return None
    if (torch.is_autocast_enabled() or not x.is_cuda or x.dim() != 2
            or x.dtype != torch.bfloat16 or not 0 < x.numel() <= NARROW_MAX_ELEMS or n > 64
            or k % 32 or x.shape[1] != k or x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16
            or first.bias is not None or second.bias is not None):
        return None
    for w in pair:
        if (w.shape != (n, k) or w.dtype != torch.bfloat16 or w.device != x.device
                or not w.is_contiguous() or w.data_ptr() % 16):
            return None
    return pair


def narrow_linears(x: torch.Tensor, first: nn.Linear, second: nn.Linear):
    """``(first(x), second(x), amax_partials)`` for two narrow bf16 linears of one
    input (``linear_attention.py:311-314``) in one ``tf_narrow_linear2`` launch,
    with max ``|x|`` per row block for ``fp8_linears`` of the same x.
    Linears that are more than plain bf16 ``nn.Linear`` calls without a bias, that
    autograd is to record or autocast to cast, or whose sizes the kernel does not
    take are called one by one (``amax_partials`` is then None)."""
    pair = _narrow_pair(x, first, second)
    if pair is None:
        return first(x), second(x), None
    n, k = pair[0].shape
    rows = x.shape[0]
    outs = [torch.empty((rows, n), dtype=torch.bfloat16, device=x.device) for _ in range(2)]
    blocks = _native.load().tf_narrow_linear2_blocks(rows)
    partials = None
    if 0 < blocks <= _native.TF_FP8_QUANT_WORKSPACE_BYTES // 4:
        partials = torch.empty((blocks,), dtype=torch.int32, device=x.device)
    _native.call("tf_narrow_linear2", _ptr(x), x.stride(0), rows, k, _ptr(pair[0]),
                 _ptr(pair[1]), n, _ptr(outs[0]), _ptr(outs[1]), n, _ptr(partials),
                 _stream_ptr(None, x.device))
    return outs[0], outs[1], partials


def fp8_linears(x: torch.Tensor, linears: Sequence["Fp8Linear"],
                amax_partials: Optional[torch.Tensor] = None):
    """``[lin(x) for lin in linears]`` for projections of the same input
    (``full_attention.py:122-139``, ``linear_attention.py:309-314``): x is
    quantised once and one GEMM launch multiplies it with every weight
    (``tf_fp8_linears``).  Linears that do not share a block size and a K that is
    a multiple of 128, or that are more than plain ``Fp8Linear`` calls, are called
    one by one.  ``amax_partials``: int32 maxima of ``|x|`` over parts of x, as
    ``narrow_linears`` leaves them (the result is the same, a pass over x less)."""
    first = linears[0]
    k = x.shape[-1]
    bh, bw = first.block_h, first.block_w
    if len(linears) <= _native.TF_FP8_MAX_MATS \
            and all(_plain(m, Fp8Linear) and m.block_h == bh and m.block_w == bw
                    for m in linears):
        x2d = x.reshape(-1, k)
        if x2d.stride(1) != 1:
            x2d = x2d.contiguous()
        weights = [(m.weight, m.weight_scale_inv, m.bias) for m in linears]
        if _takes(x2d) and all(_shared(x2d, *t, bh, bw) for t in weights):
            _check_amax(amax_partials, x2d, _native.TF_FP8_QUANT_WORKSPACE_BYTES // 4)
            outs = _linears(x2d, weights, bh, bw, amax_partials)
            return outs if x.dim() == 2 else [o.reshape(*x.shape[:-1], o.shape[1]) for o in outs]
    return [m(x) for m in linears]


class Fp8Linear(nn.Module):
    """``Qwen3_8FP8Linear`` with a float8_e4m3fn weight (``fp8_linear.py:12-212``).

    ``weight``: float8_e4m3fn ``[out_features, in_features]``;
    ``weight_scale_inv``: fp32 ``[ceil(out / block_h), ceil(in / block_w)]``
    (ones at init, like the reference), ``bias``: bf16 or absent.
    """

    def __init__(self, in_features: int, out_features: int, bias: bool = False,
                 block_size: Sequence[int] = (128, 128), device=None):
        super().__init__()
        self.in_features = in_features
        self.out_features = out_features
        self.block_h, self.block_w = int(block_size[0]), int(block_size[1])
        self.weight = nn.Parameter(
            torch.zeros((out_features, in_features), dtype=torch.float8_e4m3fn, device=device),
            requires_grad=False)
        self.register_buffer("weight_scale_inv", torch.ones(
            (math.ceil(out_features / self.block_h), math.ceil(in_features / self.block_w)),
            dtype=torch.float32, device=device), persistent=True)
        if bias:
            self.bias = nn.Parameter(torch.zeros(out_features, dtype=torch.bfloat16,
                                                 device=device), requires_grad=False)
        else:
            self.register_parameter("bias", None)

    @torch.no_grad()
    def quantize_from(self, w: torch.Tensor) -> "Fp8Linear":
        """Fills ``weight`` / ``weight_scale_inv`` from a dense ``[out, in]``
        weight with per-block scales ``amax / 448`` (the checkpoint format)."""
        out_f, in_f = self.out_features, self.in_features
        bh, bw = self.block_h, self.block_w
        wf = w.to(torch.float32)
        sh, sw = self.weight_scale_inv.shape
        pad = torch.zeros((sh * bh, sw * bw), dtype=torch.float32, device=wf.device)
        pad[:out_f, :in_f] = wf
        blocks = pad.view(sh, bh, sw, bw)
        amax = blocks.abs().amax(dim=(1, 3)).clamp(min=1e-12)
        scale = amax / FP8_MAX
        q = (blocks / scale[:, None, :, None]).clamp(-FP8_MAX, FP8_MAX)
        self.weight.copy_(q.view(sh * bh, sw * bw)[:out_f, :in_f].to(torch.float8_e4m3fn))
        self.weight_scale_inv.copy_(scale)
        return self

    def dequantize_weight(self, target_dtype: torch.dtype) -> torch.Tensor:
        """``weight * repeat_interleave(weight_scale_inv)`` (``fp8_linear.py:74-86``)."""
        scale = self.weight_scale_inv.to(torch.float32)
        full = scale.repeat_interleave(self.block_h, dim=0).repeat_interleave(self.block_w, dim=1)
        full = full[: self.out_features, : self.in_features]
        return (self.weight.to(torch.float32) * full).to(target_dtype)

    def forward(self, x: torch.Tensor, x_amax: Optional[torch.Tensor] = None) -> torch.Tensor:
        """``x_amax``: optional max ``|x|`` from x's producer (see
        ``quantize_activations``); the result does not change."""
        return block_fp8_linear(x, self.weight, self.weight_scale_inv, self.bias,
                                self.block_h, self.block_w, x_amax=x_amax)

    def extra_repr(self) -> str:
        return (f"in_features={self.in_features}, out_features={self.out_features}, "
                f"bias={self.bias is not None}, block_size=({self.block_h}, {self.block_w})")
