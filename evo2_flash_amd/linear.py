"""bf16 projections (out_proj, the attention projections, the MLP, the head):
`linear` and `gated` run on this build's weight-streaming kernel
(csrc/bf16_stream.hip) at decode batch sizes and on the platform's library GEMM
otherwise.
"""

from typing import Optional

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _lib

STREAM_ROWS = 16  # the kernel's most rows


def _eager():
    """Whether calls run as they are: nothing compiles, exports, traces or
    intercepts them (a default device apart), no autocast or forward-mode level."""
    if (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._len_torch_dispatch_stack() > 0 or torch.is_autocast_enabled("cuda")):
        return False
    if torch._C._len_torch_function_stack() > 0 and any(
            type(m) is not DeviceContext
            for m in torch.overrides._get_current_function_mode_stack()):
        return False
    return forward_ad._current_level < 0


def _ordinary(t):
    """Whether t is an ordinary dense CUDA bf16 tensor: no subclass or proxy, outside
    vmap, without a gradient to record."""
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda
            and t.layout == torch.strided and t.dtype == torch.bfloat16
            and not (t.requires_grad and torch.is_grad_enabled())
            and not torch._C._functorch.is_functorch_wrapped_tensor(t))


def plain(*tensors):
    """Whether these are ordinary CUDA bf16 matrices outside every transform (no
    tracing or dispatch mode, autocast, vmap, gradients of either mode), 16-byte
    aligned rows."""
    if not _eager():
        return False
    for t in tensors:
        if not (_ordinary(t) and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) % 8 == 0
                and t.data_ptr() % 16 == 0):
            return False
    return True


def _streams(x, *weights):
    """Whether the weight-streaming kernel takes x (M, K) against weights (N, K)."""
    # `plain` before a shape is compared: to a tracer each comparison is a
    # condition on the rows.  (x on the current device: a launch goes there, and the
    # default stream's handle is the same on every device; the library's product
    # switches over)
    return (plain(x, *weights) and 0 < x.shape[0] <= STREAM_ROWS and x.shape[1] % 32 == 0
            and x.shape[1] > 0 and all(w.shape == weights[0].shape and w.shape[0] > 0
                                       and w.shape[1] == x.shape[1]
                                       and w.stride() == weights[0].stride()
                                       and w.device == x.device for w in weights)
            and x.get_device() == torch.cuda.current_device())


def library_linear(x, weight, bias: Optional[torch.Tensor], out: Optional[torch.Tensor],
                   residual: Optional[torch.Tensor]):
    """`linear` on the library's product (also what TorchScript compiles)."""
    if out is None:
        y = torch.nn.functional.linear(x, weight, bias)
        return y if residual is None else y + residual
    if residual is not None:  # (which may be `out`: the product goes beside it)
        return torch.add(torch.nn.functional.linear(x, weight, bias), residual, out=out)
    if bias is not None:
        return torch.addmm(bias, x, weight.t(), out=out)
    return torch.mm(x, weight.t(), out=out)


def linear(x, weight, bias=None, out=None, residual=None):
    """x @ weight^T [+ bias] [+ residual], each step rounded to x's dtype; with
    `out` a 2-D x's result is written there.

    The streaming kernel takes at most 8 rows, and up to 16 of a small weight
    (N K <= 2^24, K <= 4096): there it is the faster one, measured in us against
    the library at 8 / 16 rows: 4096 x 4096 9.6 / 11.5 against 15.6; 11264 x 4096
    24.7 / 29.7 against 26.4; 1920 x 5120 11.0 / 14.3 against 18.3 / 10.5."""
    if _streams(x, weight):
        M, (N, K) = x.shape[0], weight.shape
        if ((M <= 8 or (N * K <= 1 << 24 and K <= 4096))
                and (bias is None or (_ordinary(bias) and bias.device == x.device
                                      and bias.shape == (N,) and bias.is_contiguous()))
                and (residual is None or (plain(residual) and residual.shape == (M, N)
                                          and residual.device == x.device))
                and (out is None or (_ordinary(out) and out.shape == (M, N) and out.stride(1) == 1
                                     and out.device == x.device
                                     # (the kernel stores while others still read)
                                     and not _lib.overlap(x, out)
                                     and (residual is None or not _lib.overlap(residual, out))))):
            y = torch.empty(M, N, dtype=x.dtype, device=x.device) if out is None else out
            _lib.call("evo2_bf16_stream_linear", _lib.ptr(x), x.stride(0), _lib.ptr(weight),
                      weight.stride(0), _lib.ptr(bias), _lib.ptr(residual),
                      0 if residual is None else residual.stride(0), _lib.ptr(y), y.stride(0),
                      M, N, K, _lib.stream_of(x))
            return y
    return library_linear(x, weight, bias, out, residual)


def gated(x, w1, w2, gelu):
    """act(x @ w1^T) * (x @ w2^T), act the exact GELU or the identity, each step
    rounded to x's dtype (at most 16 rows: one launch)."""
    if _streams(x, w1, w2):
        M, (N, K) = x.shape[0], w1.shape
        y = torch.empty(M, N, dtype=x.dtype, device=x.device)
        _lib.call("evo2_bf16_stream_gated", _lib.ptr(x), x.stride(0), _lib.ptr(w1), _lib.ptr(w2),
                  w1.stride(0), int(gelu), _lib.ptr(y), y.stride(0), M, N, K, _lib.stream_of(x))
        return y
    z1 = torch.nn.functional.linear(x, w1)
    z2 = torch.nn.functional.linear(x, w2)
    return (torch.nn.functional.gelu(z1) if gelu else z1) * z2


__all__ = ["linear", "gated", "plain", "STREAM_ROWS"]
