"""Projections of the models with per-sequence state."""
from __future__ import annotations

import torch.nn.functional as F
from torch import nn

from .. import ops


def linear(x, weight, bias=None):
    """F.linear; steps of few rows in 16-bit formats go through the kernel for them (ops.few_rows_product)."""
    if x.shape[0] <= ops.FEW_ROWS and ops.few_rows_fits(x, weight, bias):
        return ops.few_rows_product(x, weight, bias)
    return F.linear(x, weight, bias)


class Linear(nn.Linear):
    def forward(self, x):
        return linear(x, self.weight, self.bias)
