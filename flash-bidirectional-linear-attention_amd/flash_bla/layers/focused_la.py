"""FLatten focused linear attention (counterpart of flash_bla/layers/focused_la.py:13-96)."""
import torch.nn as nn
import torch.nn.functional as F

from flash_bla.layers import _whole
from flash_bla.layers._common import check_mode, merge_heads, torch_linear_attention
from flash_bla.layers._features import focus_formula, focused_features, merge_heads_with
from flash_bla.layers._pvt import PvtLinearAttentionBase
from flash_bla.ops.linear_attn.fused import linear_attention
from flash_bla.ops.projection import project


class FocusedLinearAttention(PvtLinearAttentionBase):
    def __init__(self, dim, num_patches, num_heads=8, qkv_bias=False, qk_scale=None, attn_drop=0., proj_drop=0.,
                 sr_ratio=1, focusing_factor=3, kernel_size=5):
        super().__init__()
        self._init_common(dim, num_patches, num_heads, qkv_bias, attn_drop, proj_drop, sr_ratio, kernel_size)
        self.q = nn.Linear(dim, dim, bias=qkv_bias)
        self.focusing_factor = focusing_factor

    def forward(self, x, H, W, mode='triton'):
        fast = check_mode(mode)
        src = self._reduced(x, H, W)
        out = _whole.focused(self, FocusedLinearAttention, x, src, H, W) if fast else None
        return self.proj_drop(self._steps(x, src, H, W, fast) if out is None else out)

    def _steps(self, x, src, H, W, fast):
        N = x.shape[1]
        kv = project(self.kv, x if src is None else src)
        features = focused_features if fast else focus_formula
        q, k, v, v_rows = features(project(self.q, x), kv, self.positional_encoding, F.softplus(self.scale),
                                   self.num_heads, self.focusing_factor)
        if fast:
            out = merge_heads_with(linear_attention(q, k, v), None, self._value_conv_tokens(v_rows, N, H, W))
        else:
            out = merge_heads(torch_linear_attention(q, k, v)) + self._value_conv(v, N, H, W)
        return project(self.proj, out)
