"""``x @ w.T (+ bias)`` with unquantised weights: a decode step's few rows on the HIP kernel that streams the weights once, everything else (prompts,
fp32, long contractions, whatever torch is to see for gradients, transforms, traces or autocast) on ``F.linear``."""
from __future__ import annotations

from typing import Optional

import torch
import torch.nn.functional as F
from torch import nn

from .. import mixer_ops as M


def project(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    if isinstance(x, torch.Tensor) and x.is_cuda and 0 < x.numel() <= 32 * x.shape[-1] and M.rows_win(x.numel() // x.shape[-1], w.shape[0], x.shape[-1]) \
            and M.outside_torch(x, w, bias):
        y = M.linear_rows(x if x.dim() == 2 else x.reshape(-1, x.shape[-1]), w, bias)
        if y is not None:
            return y if x.dim() == 2 else y.view(*x.shape[:-1], w.shape[0])
    return F.linear(x, w, bias)


def project_pair(x0: torch.Tensor, w0: torch.Tensor, x1: torch.Tensor, w1: torch.Tensor):
    """``project(x0, w0), project(x1, w1)``: of few rows and short contractions of one length in one launch."""
    if isinstance(x0, torch.Tensor) and x0.is_cuda and x0.dim() == 2 and 0 < x0.shape[0] <= 32 and M.outside_torch(x0, w0, None) and M.outside_torch(x1, w1, None):
        y = M.linear_rows_pair(x0, w0, x1, w1)
        if y is not None:
            return y
    return project(x0, w0), project(x1, w1)


class RowLinear(nn.Linear):
    """``nn.Linear`` whose product is ``project``."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return project(x, self.weight, self.bias)
