"""Dense layers of the host-side mirror (flax.linen.Dense in the reference's cells and blocks,
e.g. linear_attention.py:62-80, min_gru.py:49-62, blocks/ffn.py:11-123).

In bfloat16 over many rows the products are the library's own kernels (csrc/dense_rows.hip), and so are the
gradients (csrc/dense_grads.hip) up to the widths where those of the array library take over; there what this
module changes is their shape.  A rollout batch
has a hundred thousand rows and a few hundred features, so the weight gradient ``dy^T x`` is a
product with a tiny result and an enormous inner dimension, which the library's GEMM runs on as
many workgroups as the result has tiles (sixteen for 256 x 256: 330 us where the forward product
of the same operands takes 32 us).  Where the library's kernels do not serve a layer, ``dense`` cuts the rows
into slices, multiplies them as one batched product with float32 partial results and sums those (41 us);
``dense_group`` runs the layers that share an input on one cast of it, and their gradients as one operation.
Without gradients and on few rows (acting) the layers are one launch of the library's row kernel.  The nodes
are native (csrc/host_ops.cpp): a layer of a small update is bound by what the host does around its products.
"""
from __future__ import annotations

from typing import NamedTuple

import torch
import torch.nn as nn

from ._lib import native

_MAX_SLICES = 128   # of a weight-gradient product (csrc/host_ops.cpp)


def autocast_dtype(x):
    """The dtype the array library's autocast would run a product on ``x`` in, or None."""
    if x.is_cuda and x.is_floating_point() and torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda")
    return None


def _slices(rows, n_out, n_in):
    """Into how many slices the rows of a weight-gradient product are cut: none while the result
    has tiles enough to fill the device or the rows are few."""
    return native().weight_gradient_slices(rows, n_out, n_in)


def weight_gradient(dy, x):
    """dy^T x for dy (rows, n_out), x (rows, n_in); float32 from 16-bit operands."""
    return native().weight_gradient(dy, x)


def dense_group(x, layers):
    """The outputs of several Dense / torch.nn.Linear layers that read the same input, as a tuple.
    The layers lend their parameters; their own ``forward`` (and hooks registered on it) does not run."""
    return tuple(native().dense_group(x, [m.weight for m in layers], [m.bias for m in layers]))


def dense(x, weight, bias=None):
    """x W^T + b like torch.nn.functional.linear (autocast included), with the weight gradient as a
    sliced product (module docstring).  Gradients of weight and bias are formed in float32 when the
    operands are 16-bit and cast to the parameters' dtype by the array library."""
    return native().dense_group(x, [weight], [bias])[0]


class Dense(nn.Linear):
    """torch.nn.Linear (same parameters, same state dict) on ``dense``."""

    def forward(self, x):
        return dense(x, self.weight, self.bias)


class Weights(NamedTuple):
    """A layer that is no module: what ``dense_group`` needs of one."""
    weight: torch.Tensor
    bias: torch.Tensor | None = None
