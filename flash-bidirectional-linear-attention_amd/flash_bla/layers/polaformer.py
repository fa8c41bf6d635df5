"""PolaFormer polarity-aware linear attention (counterpart of
flash_bla/layers/polaformer.py:10-108): positive and negative parts of q, k are
kept as separate features, the same-sign and opposite-sign pairings attend to the
two halves of the value channels."""
import torch
import torch.nn as nn
import torch.nn.functional as F

from flash_bla.layers import _whole
from flash_bla.layers._common import check_mode, merge_heads, torch_linear_attention
from flash_bla.layers._features import merge_heads_with, polarity_features, polarity_formula
from flash_bla.layers._pvt import PvtLinearAttentionBase
from flash_bla.ops.linear_attn.paired import paired_linear_attention
from flash_bla.ops.projection import project


class PolaLinearAttention(PvtLinearAttentionBase):
    def __init__(self, dim, num_patches, num_heads=8, qkv_bias=False, qk_scale=None, attn_drop=0., proj_drop=0.,
                 sr_ratio=1, kernel_size=5, alpha=4):
        super().__init__()
        self.head_dim = self._init_common(dim, num_patches, num_heads, qkv_bias, attn_drop, proj_drop, sr_ratio,
                                          kernel_size)
        self.qg = nn.Linear(dim, 2 * dim, bias=qkv_bias)
        self.power = nn.Parameter(torch.zeros(1, num_heads, 1, self.head_dim))
        self.alpha = alpha

    def forward(self, x, H, W, mode='triton'):
        fast = check_mode(mode)
        src = self._reduced(x, H, W)
        out = _whole.pola(self, PolaLinearAttention, x, src, H, W) if fast else None
        return self.proj_drop(self._steps(x, src, H, W, fast) if out is None else out)

    def _steps(self, x, src, H, W, fast):
        N = x.shape[1]
        scale = F.softplus(self.scale)
        power = 1 + self.alpha * torch.sigmoid(self.power)
        # (the kernels know powers of at least 1)
        rising = isinstance(self.alpha, (int, float)) and self.alpha >= 0
        features = polarity_features if fast and rising else polarity_formula
        q_same, q_opp, k_both, v, v_rows, gate = features(project(self.qg, x), project(self.kv, x if src is None else src),
                                                          self.positional_encoding, scale, power, self.num_heads)
        if fast:  # both pairings on one state pass over the shared keys and values
            o_same, o_opp = paired_linear_attention(q_same, q_opp, k_both, v)
            out = merge_heads_with(o_same, o_opp, self._value_conv_tokens(v_rows, N, H, W), gate)
        else:
            v_same, v_opp = v.chunk(2, dim=-1)
            out = torch.cat([torch_linear_attention(q_same, k_both, v_same),
                             torch_linear_attention(q_opp, k_both, v_opp)], dim=-1)
            out = (merge_heads(out) + self._value_conv(v, N, H, W)) * gate
        return project(self.proj, out)
