"""The layer kernels of a Llama step around the paged attention
(csrc/layer_ops.hip): RMSNorm with the residual add before it, SiLU times the
up projection, and a decode step's linear layers with both folded in.

Each function has a ``*_fits`` rule: what the kernel takes. The runner asks
the modules themselves for everything else, and for any module that is not
exactly the plain one the kernel restates (a subclass, hooks, a replaced
``forward``, a bias, a tensor subclass as weight).
"""

from __future__ import annotations

import ctypes

import torch
from torch import nn
from torch.utils._device import DeviceContext

from . import _lib
from .ops import _DTYPES, _on_device, _require_backend

MAX_ROWS = _lib.DECODE_LINEAR_MAX_ROWS
# Weight elements up to which the decode linear is the faster: at 16 rows and
# 4096 x 4096 it takes 10.1 us against the library's 15.3, at 14336 x 4096
# 30 against 28.
MAX_WEIGHT = 1 << 24


def unhooked(module) -> bool:
    """True when nothing but the module's class sees a call of it."""
    return (
        not module._forward_hooks
        and not module._forward_pre_hooks
        and not module._backward_hooks
        and not module._backward_pre_hooks
        and "forward" not in module.__dict__
        and not nn.modules.module._has_any_global_hook()
    )


def plain_module(module, cls) -> bool:
    """True when calling `module` runs cls.forward and nothing else."""
    return type(module) is cls and unhooked(module)


def unwatched() -> bool:
    """True when no dispatch or function mode sees torch's calls (a flop
    counter, a tracer, a replacement for F.linear). A default device is a
    function mode too, and sees only what makes new tensors."""
    modes = (torch._C._get_function_stack_at(i) for i in range(torch._C._len_torch_function_stack()))
    return torch._C._len_torch_dispatch_stack() == 0 and all(type(m) is DeviceContext for m in modes)


def kernels_apply(x: torch.Tensor) -> bool:
    """Whether a module call on `x` may be restated by a kernel at all: no
    graph to record, no autocast, nobody watching, a plain tensor on a GPU."""
    return (
        type(x) is torch.Tensor
        and x.device.type == "cuda"
        and x.dtype in _DTYPES
        and not torch.is_grad_enabled()
        and not torch.is_autocast_enabled()
        and unwatched()
    )


def _plain_weight(w, x: torch.Tensor) -> bool:
    return (
        type(w) in (nn.Parameter, torch.Tensor)
        and w.dtype == x.dtype
        and w.device == x.device
        and w.is_contiguous()
        and w.data_ptr() % 16 == 0
    )


def _flat_rows(x: torch.Tensor) -> torch.Tensor | None:
    """`x` as [rows, cols] without a copy when its rows can be read in
    16-byte pieces, else None."""
    if x.ndim > 2:
        if not x.is_contiguous():
            return None
        x = x.view(-1, x.shape[-1])
    if x.ndim != 2 or x.stride(1) != 1 or x.data_ptr() % 16 or x.stride(0) * x.element_size() % 16:
        return None
    return x


def _stream(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


# ------------------------------------------------------------------ RMSNorm
def norm_fits(weight, x: torch.Tensor) -> bool:
    row = x.shape[-1] * x.element_size()
    return (x.numel() > 0 and row % 16 == 0 and row <= 16384 and weight.ndim == 1 and weight.shape[0] == x.shape[-1]
            and _plain_weight(weight, x) and _flat_rows(x) is not None)


def add_rms_norm(x: torch.Tensor, delta: torch.Tensor | None, weight: torch.Tensor, eps: float, *,
                 packed: bool = False):
    """(x + delta, weight * normalised rows of it); (x, ...) without delta.
    `packed`: the second in operand order, for decode_linear."""
    lib = _require_backend()
    rows = _flat_rows(x)
    out = torch.empty((MAX_ROWS, x.shape[-1]) if packed else x.shape, dtype=x.dtype, device=x.device)
    a = _lib.NormArgs()
    a.packed = packed
    a.x, a.x_stride = rows.data_ptr(), rows.stride(0)
    total = x
    if delta is not None:
        d = _flat_rows(delta)
        if d is None:  # also a contiguous one at an odd address
            d = delta.clone(memory_format=torch.contiguous_format).view(-1, delta.shape[-1])
        total = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        a.delta, a.delta_stride = d.data_ptr(), d.stride(0)
        a.sum, a.sum_stride = total.data_ptr(), x.shape[-1]
    a.weight = weight.data_ptr()
    a.out, a.out_stride = out.data_ptr(), x.shape[-1]
    a.rows, a.cols = rows.shape
    a.dtype, a.eps = _DTYPES[x.dtype], eps
    with _on_device(x.device):
        status = lib.ikl_add_rms_norm(ctypes.byref(a), _stream(x.device))
    _lib.check(status, "rms norm")
    return total, out


# --------------------------------------------------------------- SiLU * up
def silu_mul_fits(gate: torch.Tensor, up: torch.Tensor) -> bool:
    return (type(gate) is torch.Tensor and type(up) is torch.Tensor and gate.shape == up.shape
            and gate.dtype == up.dtype and gate.dtype in _DTYPES and gate.device == up.device
            and gate.device.type == "cuda" and gate.is_contiguous() and up.is_contiguous()
            and gate.numel() * gate.element_size() % 16 == 0 and (gate.data_ptr() | up.data_ptr()) % 16 == 0)


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    lib = _require_backend()
    out = torch.empty_like(gate)
    with _on_device(gate.device):
        status = lib.ikl_silu_mul(gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.numel(), _DTYPES[gate.dtype],
                                  _stream(gate.device))
    _lib.check(status, "silu mul")
    return out


# ------------------------------------------------------------ decode linears
def linear_weight_fits(linear, x: torch.Tensor) -> bool:
    """A plain bias-free 16-bit nn.Linear whose sizes are whole contraction
    steps (64) and output tiles (16)."""
    if not plain_module(linear, nn.Linear) or linear.bias is not None:
        return False
    w = linear.weight
    return (x.dtype in (torch.float16, torch.bfloat16) and w.shape[1] % 64 == 0 and w.shape[0] % 16 == 0
            and 0 < w.numel() <= MAX_WEIGHT and _plain_weight(w, x))


def linear_fits(linear, x: torch.Tensor) -> bool:
    """As linear_weight_fits, over the at most MAX_ROWS rows of `x`."""
    return (linear_weight_fits(linear, x) and x.ndim == 2 and 0 < x.shape[0] <= MAX_ROWS
            and x.shape[1] == linear.weight.shape[1] and _flat_rows(x) is not None)


def decode_linear(x: torch.Tensor, weights, *, rows: int | None = None, residual: torch.Tensor | None = None,
                  silu: bool = False, packed: bool = False):
    """x W^T for each of `weights`; with `residual` the sum, with `silu`
    silu(x W0^T) * x W1^T. One launch. `rows`: x is in operand order and has
    that many; `packed`: the result of `silu` is left in operand order."""
    lib = _require_backend()
    a = _lib.DecodeLinearArgs()
    a.x, a.x_stride, a.x_packed = x.data_ptr(), x.stride(0), rows is not None
    rows = x.shape[0] if rows is None else rows
    a.rows, a.cols = rows, x.shape[1]
    a.dtype = _DTYPES[x.dtype]
    a.num_weights = len(weights)
    outs = []
    for i, w in enumerate(weights):
        a.weight[i], a.out_cols[i] = w.data_ptr(), w.shape[0]
        if silu and i > 0:
            continue
        y = torch.empty(MAX_ROWS if packed else rows, w.shape[0], dtype=x.dtype, device=x.device)
        a.y[i], a.y_stride[i] = y.data_ptr(), w.shape[0]
        outs.append(y)
    if residual is not None:
        a.residual, a.residual_stride, a.epilogue = residual.data_ptr(), residual.stride(0), 1
    elif silu:
        a.epilogue, a.y_packed = 2, packed
    with _on_device(x.device):
        status = lib.ikl_decode_linear(ctypes.byref(a), _stream(x.device))
    _lib.check(status, "decode linear")
    return outs if len(outs) > 1 else outs[0]
