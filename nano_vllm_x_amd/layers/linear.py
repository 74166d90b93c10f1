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


def gated_rows_fit(x, proj) -> bool:
    """Whether a [gate | up] projection and its activation are one launch (ops.few_rows_glu); a hook on the projection wants it called."""
    return (x.shape[0] <= ops.FEW_ROWS and proj.bias is None and proj.weight.shape[0] % 32 == 0 and not proj._forward_hooks and not proj._forward_pre_hooks
            and ops.few_rows_fits(x, proj.weight))


class Linear(nn.Linear):
    def forward(self, x):
        return linear(x, self.weight, self.bias)
