"""nn.Linear over token rows with the weight gradient on this package's kernel.

The blocks' projections contract 1e4 to 1e5 tokens into a weight gradient of a few hundred on a side, a shape for which
the library's GEMM fills a dozen CUs; `_hip.linear_wgrad` splits the tokens and takes the bias's gradient along.  The
forward and the input's gradient stay plain library GEMMs.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from flash_bla import _hip


class TokenLinearFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.with_bias = bias is not None
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        dx = g @ weight if ctx.needs_input_grad[0] else None
        with_bias = ctx.with_bias and ctx.needs_input_grad[2]
        if torch.is_grad_enabled():  # the gradient is to be differentiated again
            rows = g.reshape(-1, g.shape[-1])
            return dx, rows.t() @ x.reshape(-1, x.shape[-1]), rows.sum(0) if with_bias else None
        dw, db = _hip.linear_wgrad(g, x, with_bias)
        return dx, dw, db


def plain_tensors(*tensors):
    """Whether these are ordinary tensors in an ordinary eager call: nothing that traces, maps, casts or carries a tangent
    through torch's own operators."""
    for t in tensors:
        if t is not None and type(t) is not torch.Tensor and type(t) is not nn.Parameter:
            return False
    return not (torch.is_autocast_enabled() or torch.compiler.is_compiling() or forward_ad._current_level >= 0 or
                torch._C._are_functorch_transforms_active())


# Results beyond these are enough tiles for the library's GEMM.  Measured in bf16, library's gradient + bias sum against the
# kernel: 1280 x 1280 over 1024 / 4096 tokens 22 + 13 against 26, 37 + 22 against 40 us; 1024 x 1024 over 2048 tokens 21 + 13
# against 24 us; 640 x 640 over 4096 tokens 29 + 19 against 21 us, 512 x 512 over 512 tokens 21 + 9 against 17 us.
MOST_WEIGHTS, MOST_WEIGHTS_WITH_BIAS = 1 << 19, 1 << 21


def splits_tokens(M, N, with_bias):
    """Whether the kernel beats the library's gradient of an M x N weight (and its bias)."""
    return M * N <= (MOST_WEIGHTS_WITH_BIAS if with_bias else MOST_WEIGHTS)


def runs_on_rows(x, weight, bias):
    """Whether the weight gradient of F.linear(x, weight, bias) is left to the kernel."""
    return (torch.is_grad_enabled() and weight.requires_grad and x.is_cuda and
            x.dtype in (torch.float16, torch.bfloat16) and weight.dtype == x.dtype and weight.device == x.device and
            (bias is None or bias.dtype == x.dtype) and x.ndim >= 2 and x.numel() > 0 and
            x.shape[-1] == weight.shape[1] and weight.shape[0] % 8 == 0 and weight.shape[1] % 8 == 0 and
            splits_tokens(*weight.shape, bias is not None) and x.numel() // x.shape[-1] <= 1 << 30 and plain_tensors(x, weight, bias))


class TokenLinear(nn.Linear):
    """nn.Linear whose backward takes the weight and bias gradients from the token-splitting kernel where that is the
    faster of the two; otherwise, and on the CPU, nn.Linear itself."""

    def forward(self, x):
        if runs_on_rows(x, self.weight, self.bias):
            return TokenLinearFunction.apply(x, self.weight, self.bias)
        return super().forward(x)
