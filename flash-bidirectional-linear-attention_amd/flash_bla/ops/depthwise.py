"""Depth-wise convolution of token rows on their H x W grid: what the vision blocks add to the attention's output
(LePE: layers/mlla.py:92, layers/rala.py:58; the value convolution: layers/focused_la.py:88-93,
layers/polaformer.py:97-101).  The reference transposes the tokens to images, runs nn.Conv2d with groups = channels and
transposes back; the kernels here read and write the tokens in place and share one filter between channels
`Cw` apart, so heads need no batch of their own.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F

from flash_bla import _hip
from flash_bla.ops._check import untouched
from flash_bla.ops.projection import gradient_of, plain_tensors


class DepthwiseConvTokensFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, H, W):
        ctx.save_for_backward(x, weight)
        ctx.grid, ctx.with_bias = (H, W), bias is not None
        return _hip.dwconv_fwd(x, weight.contiguous(), None if bias is None else bias.contiguous(), H, W)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors

        def kernels(g):
            dx = dw = db = None
            if ctx.needs_input_grad[0]:
                dx = _hip.dwconv_fwd(g, weight.contiguous(), None, *ctx.grid, flip=True)
            if ctx.needs_input_grad[1] or (ctx.with_bias and ctx.needs_input_grad[2]):
                dw, db = _hip.dwconv_grad(x, g, weight, *ctx.grid, ctx.with_bias)
            return dx, dw, db, None, None

        def composed(g):  # of torch's convolution
            bias = torch.zeros(weight.shape[0], dtype=g.dtype, device=g.device, requires_grad=True)
            with torch.enable_grad():
                inputs = [t.view_as(t) if t.requires_grad else t for t in (x, weight, bias)]
                y = _convolution_of_images(inputs[0], *ctx.grid, weight.shape[0], lambda images: F.conv2d(
                    images, *inputs[1:], padding=weight.shape[-1] // 2, groups=weight.shape[0]))
            got = iter(torch.autograd.grad(y, [t for t in inputs if t.requires_grad], g, create_graph=torch.is_grad_enabled()))
            dx, dw, db = (next(got) if t.requires_grad else None for t in inputs)
            return dx, dw, db if ctx.with_bias else None, None, None
        return gradient_of(kernels, composed, g)


def runs_on_tokens(x, conv):
    """Whether the kernels take the depth-wise nn.Conv2d `conv` on token rows x: GPU tensors of one supported type, odd
    square filters of 3 to 7 taps a side, stride 1, "same" zero padding, whole 16-byte pieces of channels; a module
    without hooks."""
    K = conv.kernel_size[0]
    w, bias = conv.weight, conv.bias
    Cw = w.shape[0]
    return (untouched(conv, nn.Conv2d) and plain_tensors(x, w, bias) and x.is_cuda and x.numel() > 0 and
            x.dtype in (torch.float16, torch.bfloat16, torch.float32) and w.dtype == x.dtype and w.device == x.device and
            (bias is None or bias.dtype == x.dtype and bias.device == x.device and bias.numel() == Cw) and
            K in (3, 5, 7) and conv.kernel_size == (K, K) and w.shape == (Cw, 1, K, K) and
            conv.padding == (K // 2, K // 2) and conv.padding_mode == 'zeros' and conv.stride == (1, 1) and
            conv.dilation == (1, 1) and conv.groups == Cw and
            x.shape[-1] % Cw == 0 and x.shape[-1] % (16 // x.element_size()) == 0)


def depthwise_conv_tokens(x, conv, H, W):
    """The depth-wise convolution `conv` (an nn.Conv2d over Cw channels) of token rows x [B, H*W, C], C a multiple of
    Cw: channel c is convolved with filter c % Cw.  Returns [B, H*W, C].  What the kernels do not take (CPU tensors,
    other filter shapes, an H or W that the tokens do not fill: the reshape there refuses it) runs as the torch
    convolution of the transposed tokens."""
    if x.shape[1] == H * W and runs_on_tokens(x, conv):
        return DepthwiseConvTokensFunction.apply(x, conv.weight, conv.bias, H, W)
    return _convolution_of_images(x, H, W, conv.weight.shape[0], conv)


def _convolution_of_images(x, H, W, Cw, convolve):
    B, N, C = x.shape
    images = x.reshape(B, H, W, C // Cw, Cw).permute(0, 3, 4, 1, 2).reshape(B * (C // Cw), Cw, H, W)
    return convolve(images).reshape(B, C, N).transpose(1, 2)
