"""nn.Linear whose few-row calls run the weight-streaming skinny kernel.

The decoder's projections (the reference's QKVParallelLinear, RowParallelLinear,
MergedColumnParallelLinear and ParallelLMHead, layers/linear.py, layers/embed_head.py,
on one GPU) are plain linear layers; in a decode step they see one row per
sequence, and streaming the weights is the whole cost.  Calls with at most 16
rows that vlc_linear_skinny takes run there; calls of 17 to 64 rows on a weight at least
four times as long as it is tall run in vlc_linear_split (the down projections: 18944 x 3584
with 32 rows 38 us against the library's 110, 11008 x 2048 18 against 27; on the other
projections, where K is at most N, the library is the faster one from 17 rows on, 3584 x
37888 57 against 82 us).  On such weights 65 to 2500 rows run in vlc_linear_tiled (18944 x 3584
with 100 rows 38 us against 98, 1247 rows 169 against 227, 11008 x 2048 23 against 30 and 72
against 87; the library is ahead at 18944 x 3584 with 1600 rows, 225 against 245, and at 11008 x 2048 from
3000 rows on).  Every other call is torch's F.linear (hipBLASLt).
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import nn

from .. import kernels


class Linear(nn.Linear):

    def forward(self, x):
        x2 = x if x.dim() == 2 else x.reshape(-1, x.shape[-1])
        if x2.shape[0] <= kernels.SKINNY_MAX_ROWS and kernels.linear_skinny_supported(x2, self.weight, self.bias):
            y = kernels.linear_skinny(x2, self.weight, self.bias)
            return y if x.dim() == 2 else y.view(*x.shape[:-1], y.shape[-1])
        # F.linear records a graph for its backward; these kernels do not
        rows = x2.shape[0]
        if kernels.SKINNY_MAX_ROWS < rows <= kernels.TILED_MAX_ROWS and self.in_features >= 4 * self.out_features and \
                not torch.is_grad_enabled():
            if rows <= kernels.SPLIT_MAX_ROWS and kernels.linear_split_supported(x2, self.weight, self.bias):
                y = kernels.linear_split(x2, self.weight, self.bias)
                return y if x.dim() == 2 else y.view(*x.shape[:-1], y.shape[-1])
            if rows > kernels.SPLIT_MAX_ROWS and kernels.linear_tiled_supported(x2, self.weight, self.bias):
                y = kernels.linear_tiled(x2, self.weight, self.bias)
                return y if x.dim() == 2 else y.view(*x.shape[:-1], y.shape[-1])
        return F.linear(x, self.weight, self.bias)


kernels._LINEAR_FORWARDS.add(Linear.forward)
