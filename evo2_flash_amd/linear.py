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
_TENSORS = (torch.Tensor, torch.nn.Parameter)


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
    return (type(t) in _TENSORS and t.is_cuda
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
    # what traces comes before a shape is compared: to a tracer each comparison is
    # a condition on the rows.  (Most rows go to the library: their count comes
    # next.)
    if (type(x) not in _TENSORS or torch.compiler.is_compiling() or torch.jit.is_tracing()
            or x.dim() != 2 or not 0 < x.shape[0] <= STREAM_ROWS):
        return False
    # (x on the current device: a launch goes there, and the default stream's
    # handle is the same on every device; the library's product switches over)
    return (plain(x, *weights) and x.shape[1] % 32 == 0 and x.shape[1] > 0
            and all(w.shape == weights[0].shape and w.shape[0] > 0
                    and w.shape[1] == x.shape[1] and w.stride() == weights[0].stride()
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


def stream_rows(N, K, residual=False):
    """The most rows for which the streaming kernel is the faster one of an
    (N, K) weight.  The library's time hardly depends on the rows; the kernel's
    grows with rows x K, which every 16 columns' workgroup reads from the L2.
    Weights from HBM, us against the library's: 4096 x 4096 9.6 at 8 rows and
    11.6 at 16 against 15.5; 11264 x 4096 24.8 and 30.1 against 26.3; 1920 x 5120
    10.8 and 14.4 against 18.2 and 10.3; 24576 x 8192 77.2 at 4 and 85.2 at 8
    against 80.9 and 78.8; 4096 x 11264 19.6 and 20.5 against 20.8 and 19.8, and
    22.4 against 22.0 where the library's residual takes another launch (8192 x
    11264 then 40.7 against 37.3); behind it at 1 to 8 rows 6144 x 6144 (20.9 - 23.4
    against 19), 512 x 8192 from 2 rows (14.2 at 8 against 11.5), 8192 x 22528 from
    3 (81 at 8 against 71)."""
    if K <= 5120:
        return 16 if N * K <= 1 << 24 and K <= 4096 else 8
    if 8192 <= K <= 11264 and N >= 4096:
        return 8 if residual and N * K <= 1 << 26 else 4
    return 0


def gated_rows(K):
    """The most rows for which `gated` streams: 11264 x 4096 46.4 us at 16 against
    the library's 53.2 in three launches; 22528 x 8192 146.7 at 8 against 149.4,
    153.3 at 10 against 150.3; 4096 x 16384 behind it from one row (72.5, 61.9)."""
    return 16 if K <= 5120 else 8 if K <= 11264 else 0


def linear(x, weight, bias=None, out=None, residual=None):
    """x @ weight^T [+ bias] [+ residual], each step rounded to x's dtype; with
    `out` a 2-D x's result is written there.  Up to stream_rows rows on the
    streaming kernel."""
    if _streams(x, weight):
        M, (N, K) = x.shape[0], weight.shape
        if (M <= stream_rows(N, K, residual is not None)
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
    rounded to x's dtype (up to gated_rows rows: one launch)."""
    if _streams(x, w1, w2) and x.shape[0] <= gated_rows(x.shape[1]):
        M, (N, K) = x.shape[0], w1.shape
        y = torch.empty(M, N, dtype=x.dtype, device=x.device)
        _lib.call("evo2_bf16_stream_gated", _lib.ptr(x), x.stride(0), _lib.ptr(w1), _lib.ptr(w2),
                  w1.stride(0), int(gelu), _lib.ptr(y), y.stride(0), M, N, K, _lib.stream_of(x))
        return y
    z1 = torch.nn.functional.linear(x, w1)
    z2 = torch.nn.functional.linear(x, w2)
    return (torch.nn.functional.gelu(z1) if gelu else z1) * z2


__all__ = ["linear", "gated", "plain", "STREAM_ROWS"]
