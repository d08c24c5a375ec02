"""MLP block and channel LayerNorm with the reference's names and parameters
(segment_anything_fast/modeling/common.py:13-43).  lin1 / lin2 are ordinary
nn.Linear modules so that quant.apply_dynamic_quant can swap them."""

from typing import Type

import torch
import torch.nn as nn

from .. import ops


class MLPBlock(nn.Module):
    def __init__(self, embedding_dim: int, mlp_dim: int, act: Type[nn.Module] = nn.GELU) -> None:
        super().__init__()
        self.lin1 = nn.Linear(embedding_dim, mlp_dim)
        self.lin2 = nn.Linear(mlp_dim, embedding_dim)
        self.act = act()

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.lin2(self.act(self.lin1(x)))


class LayerNorm2d(nn.Module):
    """LayerNorm over the channel axis of (B, C, H, W).  Channels-last half-type input on a GPU without
    autograd (what the encoder's neck sees) is one launch over its rows of C values, statistics in
    fp32; anything else is composed from tensor operations."""

    def __init__(self, num_channels: int, eps: float = 1e-6) -> None:
        super().__init__()
        self.weight = nn.Parameter(torch.ones(num_channels))
        self.bias = nn.Parameter(torch.zeros(num_channels))
        self.eps = eps

    def _rows_ok(self, x: torch.Tensor) -> bool:
        return (x.is_cuda and x.dim() == 4 and x.dtype in (torch.bfloat16, torch.float16) and not torch.is_grad_enabled()
                and self.weight.dtype == x.dtype and self.bias.dtype == x.dtype and self.eps >= 0
                and x.shape[1] == self.weight.numel() and x.shape[1] % 8 == 0 and x.shape[1] <= 4096
                and ops.unwatched(x) and ops.rows_launchable(x.permute(0, 2, 3, 1), self.weight, self.bias))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if self._rows_ok(x):
            return ops.layernorm(x.permute(0, 2, 3, 1), self.weight, self.bias, self.eps).permute(0, 3, 1, 2)
        mean = x.mean(1, keepdim=True)
        centered = x - mean
        var = centered.pow(2).mean(1, keepdim=True)
        y = centered / torch.sqrt(var + self.eps)
        return y * self.weight[:, None, None] + self.bias[:, None, None]
