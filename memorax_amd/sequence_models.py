"""Host-side mirror of memorax's sequence-model interface, on top of the HIP kernels.

Same contract as the reference (memorax/networks/sequence_models):

    SequenceModel.__call__(inputs (B,T,F), done (B,T), initial_carry=None) -> (next_carry, y)
    SequenceModel.initialize_carry(key, input_shape=(B,F)) -> carry          sequence_model.py:8-19
    MemoroidCellBase: __call__(x) -> elements, binary_operator(a, b), read(h, x),
                      initialize_carry(key, input_shape)                      memoroid.py:20-33
    Memoroid(cell)(inputs, done, initial_carry) = read(scan(cell(inputs)))    memoroid.py:93-109

Carries keep the reference's pytree shapes (leaves with a size-1 time axis, (B,1,...)),
so Stack-style per-block carry tuples and checkpointing keep working.

What differs: the reference scans *any* cell algebra with jax.lax.associative_scan
(memoroid.py:60-91).  Here each cell also implements ``scan(elements, carry, done)``,
which hands its algebra to the matching fused kernel (diagonal scan, chunked linear
attention, chunked delta rule) instead of materialising per-step states;
``binary_operator`` remains the definition of the algebra (and is what the tests fold
to check ``scan``).  Modules are torch.nn.Modules: torch plays the role of the array
library / autodiff host here, the arithmetic of the recurrences runs in the kernels.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from typing import NamedTuple

from torch.nn.modules.module import _has_any_global_hook as _any_global_hook

from ._lib import native
from .dense import Dense, Weights, autocast_dtype, dense, dense_group
from .functional import (deltanet, gated_linear_attention, linear_attention, linear_scan, mingru_scan, mlstm_gates,
                         normalised_linear_attention, layer_norm, layer_norm_fork, rms_norm, rms_norm_fork, silu_gate,
                         stepping_in_place)
from .kernels import RMS_NORM_MAX_D as _RMS_NORM_MAX_D


# ----------------------------------------------------------------------------------
# axes helpers (memorax/utils/axes.py:19-32,46-49)
# ----------------------------------------------------------------------------------
def add_time_axis(x):
    return x[:, None]


def remove_time_axis(x):
    return x.squeeze(1)


def get_input_shape(inputs):
    """(B, T, F) -> (B, F)."""
    return inputs.shape[:1] + inputs.shape[2:]


class SequenceModel(nn.Module):
    """sequence_model.py:8-19."""

    def forward(self, inputs, done, initial_carry=None, **kwargs):  # pragma: no cover
        raise NotImplementedError

    def initialize_carry(self, key, input_shape):  # pragma: no cover
        raise NotImplementedError

    def acting(self, x, norm, done, carry):
        """The pre-norm residual block around this model for one acting step; see MemoroidCellBase.acting."""
        return None

    def onto(self, residual, inputs, done, carry):
        """(next_carry, residual + y) where the model's last layer takes the sum with it; else None."""
        return None


class MemoroidCellBase(nn.Module):
    """memoroid.py:20-33 plus the kernel hook ``scan``."""

    def forward(self, x, **kwargs):  # elements
        raise NotImplementedError

    def binary_operator(self, a, b):
        raise NotImplementedError

    def read(self, h, x, **kwargs):
        raise NotImplementedError

    def initialize_carry(self, key, input_shape):
        raise NotImplementedError

    def whole(self, x, done, initial_carry):
        """read(scan(self(x))) as one operation, (next_carry, y), where a cell has it for these arrays; else None."""
        return None

    def whole_onto(self, residual, x, done, initial_carry):
        """(next_carry, residual + y) with y as ``whole`` forms it, where a cell's last product takes the sum with it; else None.
        initial_carry: None where the cell is to make it."""
        return None

    def acting(self, x, norm, done, carry):
        """(next_carry, x + read(scan(self(norm(x))))) for one time step without gradients (``_acts``), where a cell has its
        launches fused for these arrays; else None."""
        return None

    def closes(self):
        """Whether ``closing`` stands for this cell's read-out."""
        return False

    def closing(self, h, x):
        """(layer, rows): read(h, x) is the dense layer ``layer`` on ``rows``."""
        raise NotImplementedError

    def scan(self, z, initial_carry, done):
        """Reset-aware inclusive scan of the cell's algebra over time, carry-in
        prepended (memoroid.py:60-91).  Returns (h, next_carry).

        The cells of this module override it with a fused kernel.  This default serves any other
        cell that only defines ``binary_operator``: the same scan with array operations, on whatever
        device the elements live on (``generic_scan``)."""
        return generic_scan(self.binary_operator, z, initial_carry, done)


def _tree_map(fn, tree, *rest):
    """fn over the leaves of nested tuples / lists / dicts (named tuples keep their type)."""
    if isinstance(tree, dict):
        return {k: _tree_map(fn, v, *(r[k] for r in rest)) for k, v in tree.items()}
    if isinstance(tree, (tuple, list)):
        out = [_tree_map(fn, v, *(r[i] for r in rest)) for i, v in enumerate(tree)]
        return type(tree)(*out) if hasattr(tree, "_fields") else type(tree)(out)
    return fn(tree, *rest)


def broadcast_done(done, carry):
    """utils/axes.py:64-68: trailing axes added to (or dropped from) done until its rank is the leaf's."""
    while done.dim() != carry.dim():
        done = done[..., None] if done.dim() < carry.dim() else done[..., 0]
    return done


def generic_scan(binary_operator, z, initial_carry, done):
    """Memoroid.scan_fn (memoroid.py:60-91) for an arbitrary pytree algebra.

    The carry becomes slot 0 of every leaf with reset flag 0; slots are combined with the augmented
    operator ``(where(reset_b, b, a (+) b), max(reset_a, reset_b))`` -- the right element wins by
    *select* when its reset flag is set -- and the result is split into the T prefixes and the last
    one (time axis of size 1).  Instead of jax.lax.associative_scan's odd/even recursion the slots
    are combined by doubling: ceil(log2(T + 1)) rounds, each one call of ``binary_operator`` on leaves
    of shape (B, n, ...) (n slots at once; the reference maps the operator over B, so it sees
    (n, ...)); there is no host loop over time steps, and autograd differentiates through it.
    Leaves are (B, T, ...); ``done`` is (B, T), bool or float."""
    zz = _tree_map(lambda c, e: torch.cat([c, e], dim=1), initial_carry, z)
    first = zz
    while isinstance(first, (tuple, list, dict)):
        first = next(iter(first.values())) if isinstance(first, dict) else first[0]
    reset = torch.cat([done.new_zeros((done.shape[0], 1), dtype=torch.bool), done != 0], dim=1)[..., None]
    n, shift = first.shape[1], 1
    while shift < n:
        left = _tree_map(lambda x: x[:, :-shift], zz)
        right = _tree_map(lambda x: x[:, shift:], zz)
        rr = reset[:, shift:]
        comb = binary_operator(left, right)
        comb = _tree_map(lambda r, c: torch.where(broadcast_done(rr, r), r, c), right, comb)
        zz = _tree_map(lambda x, c: torch.cat([x[:, :shift], c], dim=1), zz, comb)
        reset = torch.cat([reset[:, :shift], reset[:, :-shift] | rr], dim=1)
        shift *= 2
    return _tree_map(lambda x: x[:, 1:], zz), _tree_map(lambda x: x[:, -1:], zz)


class Memoroid(SequenceModel):
    """memoroid.py:57-112 (without the RTRL hooks).  The cells of this module scan with their fused
    kernels: the matrix-state cells (linear attention, Mamba, mLSTM) put the query among their elements,
    because their kernels fuse the read-out contraction into the scan, so that ``scan`` returns the
    carry like any other cell's.  Any other MemoroidCellBase -- a user's cell that defines only
    ``binary_operator`` -- is scanned by the base class's generic ``scan``, as the reference scans
    every cell."""

    def __init__(self, cell: MemoroidCellBase):
        super().__init__()
        self.cell = cell

    def forward(self, inputs, done, initial_carry=None, **kwargs):
        if initial_carry is None:
            initial_carry = self.cell.initialize_carry(None, get_input_shape(inputs))
        whole = None if kwargs or _hooked(self.cell) else self.cell.whole(inputs, done, initial_carry)
        if whole is not None:
            return whole
        z = self.cell(inputs, **kwargs)
        h, next_carry = self.cell.scan(z, initial_carry, done)
        y = self.cell.read(h, inputs, **kwargs)
        return next_carry, y

    def onto(self, residual, inputs, done, carry):
        if type(self).forward is not Memoroid.forward:
            return None
        if type(self.cell).whole is not MemoroidCellBase.whole:
            return self.cell.whole_onto(residual, inputs, done, carry)
        if not self.cell.closes():
            return None
        if carry is None:
            carry = self.cell.initialize_carry(None, get_input_shape(inputs))
        h, next_carry = self.cell.scan(self.cell(inputs), carry, done)
        layer, rows = self.cell.closing(h, inputs)
        return next_carry, native().dense_onto(residual, rows, layer.weight, layer.bias)

    def acting(self, x, norm, done, carry):
        if type(self).forward is not Memoroid.forward:
            return None
        return self.cell.acting(x, norm, done, self.cell.initialize_carry(None, get_input_shape(x)) if carry is None else carry)

    def initialize_carry(self, key, input_shape):
        return self.cell.initialize_carry(key, input_shape)


# ----------------------------------------------------------------------------------
# diagonal algebra cells
# ----------------------------------------------------------------------------------
class _DiagonalCell(MemoroidCellBase):
    """Cells whose elements are (state, decay) with
    binary_operator(a, b) = (decay_b * state_a + state_b, decay_b * decay_a)
    (lru.py:92-95, s5.py:133-136).  ``scan`` returns h = (states (B,T,N), None): the
    per-step cumulative decay is never materialised, only its last value (the carry)."""

    def binary_operator(self, a, b):
        state_i, decay_i = a
        state_j, decay_j = b
        return (decay_j * state_i + state_j, decay_j * decay_i)

    def scan(self, z, initial_carry, done):
        state, decay = z            # decay: (B,T,N) or time-invariant (N,)
        h0, P0 = initial_carry      # (B,1,N)
        h, h_last, P_last = linear_scan(decay, state, done, h0[:, 0].contiguous(), P0[:, 0].contiguous())
        return (h, None), (h_last[:, None], P_last[:, None])


def _complex_states(x, weight):
    """x B^T for real x (B,T,F) and complex B given as (N, 2, F) (real and imaginary rows): one real product whose columns are
    the complex result's components.  A complex product of x with a zero imaginary part is four times the arithmetic, and its
    weight gradient -- a small complex result over every row -- took nine tenths of an LRU layer's update."""
    N = weight.shape[0]
    with torch.autocast(x.device.type, enabled=False):   # the recurrence runs in complex64 whatever surrounds it
        out = dense(x.float(), weight.reshape(2 * N, -1).float())
    return torch.view_as_complex(out.view(*out.shape[:-1], N, 2))


def _real_read_out(state, weight):
    """Re(state C^T) for complex state (B,T,N), C given as (F, N, 2) with (Re C, -Im C): one real product."""
    flat = torch.view_as_real(state).flatten(-2)
    with torch.autocast(state.device.type, enabled=False):
        return dense(flat, weight.flatten(-2).to(flat.dtype))


class LRUCell(_DiagonalCell):
    """Linear Recurrent Unit, complex diagonal recurrence (lru.py:32-108).  The decay
    lambda is time-invariant and is passed to the kernel as an (N,) vector instead of
    being broadcast to (B,T,N) (lru.py:86)."""

    def __init__(self, features, hidden_dim, r_min=0.0, r_max=1.0, max_phase=6.28):
        super().__init__()
        self.features, self.hidden_dim = features, hidden_dim
        u1, u2 = torch.rand(hidden_dim), torch.rand(hidden_dim)
        nu_log = torch.log(-0.5 * torch.log(u1 * (r_max**2 - r_min**2) + r_min**2))   # lru.py:12-14
        theta_log = torch.log(max_phase * u2)                                          # lru.py:17-19
        lam = torch.exp(-torch.exp(nu_log) + 1j * torch.exp(theta_log))
        self.nu_log = nn.Parameter(nu_log)
        self.theta_log = nn.Parameter(theta_log)
        self.gamma_log = nn.Parameter(torch.log(torch.sqrt(1 - torch.abs(lam) ** 2)))  # lru.py:22-25
        self.B_real = nn.Parameter(torch.randn(hidden_dim, features) / math.sqrt(2 * features))
        self.B_imag = nn.Parameter(torch.randn(hidden_dim, features) / math.sqrt(2 * features))
        self.C_real = nn.Parameter(torch.randn(features, hidden_dim) / math.sqrt(hidden_dim))
        self.C_imag = nn.Parameter(torch.randn(features, hidden_dim) / math.sqrt(hidden_dim))
        self.D = nn.Parameter(torch.randn(features))

    def forward(self, x, **kwargs):
        lam = torch.polar(torch.exp(-torch.exp(self.nu_log)), torch.exp(self.theta_log))
        return (_complex_states(x, torch.stack([self.B_real, self.B_imag], 1) * torch.exp(self.gamma_log)[:, None, None]), lam)

    def read(self, h, x, **kwargs):
        return _real_read_out(h[0], torch.stack([self.C_real, -self.C_imag], -1)) + self.D * x

    def _parameters_in_order(self):
        return [self.nu_log, self.theta_log, self.gamma_log, self.B_real, self.B_imag, self.C_real, self.C_imag, self.D]

    def whole(self, x, done, initial_carry):
        """The layer as one native operation (lru_cells.hip around the products and the scan) where gradients are recorded: float32 on the
        device, rows of whole vectors.  Of the composition's array operations two thirds make and differentiate small matrices of parameters."""
        return self._layer(None, x, done, initial_carry)

    def whole_onto(self, residual, x, done, initial_carry):
        return self._layer(residual, x, done, initial_carry) if type(self).whole is LRUCell.whole else None

    def _layer(self, residual, x, done, initial_carry):
        params = self._parameters_in_order()
        if not (torch.is_grad_enabled() and _as_written(self, LRUCell) and x.is_cuda and x.dtype is torch.float32 and x.dim() == 3
                and autocast_dtype(x) is None and x.shape[0] * x.shape[1] >= _SPLIT_TERMS <= self.features and 2 * self.hidden_dim >= _SPLIT_TERMS
                and x.shape[2] == self.features and self.features % 8 == 0 and self.hidden_dim % 4 == 0 and 2 * self.hidden_dim * self.features <= 1 << 20
                and all(p.dtype is torch.float32 for p in params)):
            return None
        h0, P0 = self.initialize_carry(None, get_input_shape(x)) if initial_carry is None else initial_carry
        y, h, P = native().lru_layer(x, residual, params, done, h0[:, 0], P0[:, 0])
        return (h[:, None], P[:, None]), y

    def acting(self, x, norm, done, carry):
        params = self._parameters_in_order()
        # fused / composed, in a graph and host-issued (us, features = hidden width): 1024 x 512 64 / 75 and 61 / 146, 4096 x 512 190 / 142 and
        # 180 / 147, 256 x 1024 66 / 78 and 64 / 146, 1024 x 1024 227 / 133 and 213 / 145
        if not (_as_written(self, LRUCell) and autocast_dtype(x) is None and self.hidden_dim % 8 == 0 and 2 * self.hidden_dim <= _RMS_NORM_MAX_D
                and x.shape[0] * self.features * self.hidden_dim <= 1 << 28 and all(p.dtype is torch.float32 for p in params)):
            return None
        y, *carry = native().lru_act(x, *_norm_of(norm), params, done, *carry)
        return tuple(carry), y

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.nu_log.device
        return (torch.zeros(*batch, 1, self.hidden_dim, dtype=torch.complex64, device=dev),
                torch.ones(*batch, 1, self.hidden_dim, dtype=torch.complex64, device=dev))


def _dplr_hippo(n):
    """Eigenvalues and eigenvectors of the normal part of the HiPPO-LegS matrix
    (networks/hippo.py:6-37), in float64 NumPy."""
    import numpy as np
    p = np.sqrt(1.0 + 2.0 * np.arange(n))
    a = -(np.tril(p[:, None] * p[None, :]) - np.diag(np.arange(n)))
    pl = np.sqrt(np.arange(n) + 0.5)
    sm = a + pl[:, None] * pl[None, :]
    lam_real = np.full(n, np.mean(np.diag(sm)))
    lam_imag, v = np.linalg.eigh(sm * (-1j))
    return lam_real + 1j * lam_imag, v


class S5Cell(_DiagonalCell):
    """S5: diagonal state space model with HiPPO-N initialised eigenvalues, discretised with a
    learned per-state step (s5.py:28-149).  As for the LRU the discretised decay is time-invariant
    and goes to the kernel as an (N,) vector instead of being broadcast (s5.py:127)."""

    def __init__(self, features, state_size, discretization="zoh", dt_min=0.001, dt_max=0.1,
                 clip_eigens=False, step_rescale=1.0):
        super().__init__()
        import numpy as np
        self.features, self.state_size = features, state_size
        self.discretization, self.clip_eigens, self.step_rescale = discretization, clip_eigens, step_rescale
        lam, v = _dplr_hippo(state_size)
        v_inv = torch.from_numpy(v.conj().T.copy())
        vt = torch.from_numpy(v.copy())
        self.lambda_real = nn.Parameter(torch.from_numpy(lam.real.copy()).float())
        self.lambda_imag = nn.Parameter(torch.from_numpy(lam.imag.copy()).float())
        b = (v_inv @ (torch.randn(state_size, features, dtype=torch.float64) / math.sqrt(features)).to(v_inv.dtype))
        c = (torch.randn(features, state_size, dtype=torch.float64).clamp(-2, 2).to(vt.dtype) @ vt)
        self.B = nn.Parameter(torch.stack([b.real, b.imag], -1).float())     # (N, F, 2)
        self.C = nn.Parameter(torch.stack([c.real, c.imag], -1).float())     # (F, N, 2)
        self.d = nn.Parameter(torch.randn(features))
        self.log_step = nn.Parameter(torch.rand(state_size, 1) * (math.log(dt_max) - math.log(dt_min)) + math.log(dt_min))

    def _discretized_params(self):
        lr = torch.clamp(self.lambda_real, max=-1e-4) if self.clip_eigens else self.lambda_real
        lam = torch.complex(lr, self.lambda_imag)
        b_tilde = torch.complex(self.B[..., 0], self.B[..., 1])
        c_tilde = torch.complex(self.C[..., 0], self.C[..., 1])
        step = (self.step_rescale * torch.exp(self.log_step[:, 0])).to(torch.complex64)
        if self.discretization == "zoh":          # hippo.py:51-57
            lambda_bar = torch.exp(lam * step)
            b_bar = ((lambda_bar - 1.0) / lam)[:, None] * b_tilde
        elif self.discretization == "bilinear":   # hippo.py:40-48
            bl = 1.0 / (1.0 - (step / 2.0) * lam)
            lambda_bar = bl * (1.0 + (step / 2.0) * lam)
            b_bar = (bl * step)[:, None] * b_tilde
        else:
            raise ValueError(f"Invalid discretization: {self.discretization}")
        return lambda_bar, b_bar, c_tilde

    def forward(self, x, **kwargs):
        lambda_bar, b_bar, _ = self._discretized_params()
        return (_complex_states(x, torch.view_as_real(b_bar).transpose(1, 2)), lambda_bar.to(torch.complex64))

    def read(self, h, x, **kwargs):   # c_tilde is C as it is learned: (F, N, 2)
        return _real_read_out(h[0], torch.stack([self.C[..., 0], -self.C[..., 1]], -1)) + self.d * x

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.d.device
        return (torch.zeros(*batch, 1, self.state_size, dtype=torch.complex64, device=dev),
                torch.ones(*batch, 1, self.state_size, dtype=torch.complex64, device=dev))


class _SownValues(dict):
    """What the reference records with flax's ``sow`` (min_gru.py:63): the value is formed when it is read,
    not when it is recorded -- a mean over a (B,T,F) array is a pass over memory that a training step never
    looks at.  Until then the entry holds on to the array it will be formed from."""

    def sow(self, name, thunk):
        dict.__setitem__(self, name, thunk)

    def __getitem__(self, name):
        value = dict.__getitem__(self, name)
        if callable(value):
            value = value()
            dict.__setitem__(self, name, value)
        return value


def _gated(value, gate):
    """value * silu(gate) (blocks/ffn.py:108-121 with silu): the library's kernel on the device."""
    return silu_gate(value, gate) if gate.is_cuda else value * F.silu(gate)


class MinGRUProjections(NamedTuple):
    """MinGRU's elements before the element map: the step's two projections.  ``MinGRUCell.scan``
    hands them to the kernel that applies the map (a = sigma(-z), b = sigma(z) g(h~)) itself."""
    z: torch.Tensor
    h_tilde: torch.Tensor


class MinGRUCell(_DiagonalCell):
    """MinGRU (min_gru.py:14-90).  The reference scans (log_state, log_decay) with
    logaddexp; the same recurrence in linear space is h_t = sigma(-z) h_{t-1} +
    sigma(z) g(h~), g(x) = x + 0.5 (x >= 0) | sigma(x), which is what the kernel scans.
    The carry keeps the reference's log-space leaves: (log h_T, sum of log decays).
    fused (default): the cell returns the projections and the scan kernel forms the coefficients,
    so neither they nor the half dozen elementwise intermediates behind them exist in memory;
    fused=False returns the linear-space elements (b, a) for the generic diagonal scan."""

    def __init__(self, features, in_features=None, fused=True):
        super().__init__()
        self.features, self.fused = features, fused
        in_features = features if in_features is None else in_features
        self.z = Dense(in_features, features, bias=False)
        self.h = Dense(in_features, features, bias=False)
        self.intermediates = _SownValues()

    def forward(self, x, **kwargs):
        return self.elements(*dense_group(x, [self.z, self.h]))

    def elements(self, z, h_tilde):
        """The cell's elements from its two projections."""
        self.intermediates.sow("gate", lambda z=z.detach(): z.float().mean())   # min_gru.py:63 sows the mean gate
        if self.fused:   # the recurrence runs in fp32 whatever the projections' dtype (autocast): the kernels
            # read bfloat16 projections as they are (and write bfloat16 states); anything else goes in as float32
            if z.dtype == torch.bfloat16 and h_tilde.dtype == torch.bfloat16:
                return MinGRUProjections(z, h_tilde)
            return MinGRUProjections(z.float(), h_tilde.float())
        z, h_tilde = z.float(), h_tilde.float()
        a = torch.sigmoid(-z)
        g = torch.where(h_tilde >= 0, torch.relu(h_tilde) + 0.5, torch.sigmoid(h_tilde))
        return ((torch.sigmoid(z) * g).contiguous(), a.contiguous())

    def scan(self, z, initial_carry, done):
        log_state, log_decay = initial_carry
        h0, P0 = torch.exp(log_state), torch.exp(log_decay)
        if isinstance(z, MinGRUProjections):
            h, h_last, P_last = mingru_scan(z.z, z.h_tilde, done, h0[:, 0].contiguous(), P0[:, 0].contiguous())
            h_last, P_last = h_last[:, None], P_last[:, None]
        else:
            (h, _), (h_last, P_last) = super().scan(z, (h0, P0), done)
        return (h, None), (torch.log(h_last), torch.log(P_last))

    def read(self, h, x, **kwargs):
        return h[0]

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.z.weight.device
        return (torch.full((*batch, 1, self.features), -math.inf, device=dev),
                torch.zeros(*batch, 1, self.features, device=dev))


class GatedLinearRecurrence(SequenceModel):
    """Gated MLP whose hidden activation is a MinGRU-style diagonal recurrence:
    y = W_o( scan(a = sigma(-W_z x), b = sigma(W_z x) g(W_h x)) * silu(W_g x) ),
    i.e. the recurrence of min_gru.py:49-78 inside the gating pattern of the reference's GLU
    block (blocks/ffn.py:82-123).  Carry = MinGRUCell's (log_state, log_decay)."""

    def __init__(self, features, hidden=None):
        super().__init__()
        hidden = features if hidden is None else hidden
        self.cell = MinGRUCell(hidden, in_features=features)
        self.gate = Dense(features, hidden, bias=False)
        self.out = Dense(hidden, features, bias=False)

    def forward(self, inputs, done, initial_carry=None, **kwargs):
        if initial_carry is None:
            initial_carry = self.cell.initialize_carry(None, get_input_shape(inputs))
        rows, next_carry = self._gated_states(inputs, done, initial_carry)
        return next_carry, self.out(rows)

    def _gated_states(self, inputs, done, carry):
        z, h_tilde, gate = dense_group(inputs, [self.cell.z, self.cell.h, self.gate])
        h, next_carry = self.cell.scan(self.cell.elements(z, h_tilde), carry, done)
        return _gated(h[0], gate), next_carry

    def onto(self, residual, inputs, done, carry):
        if not (type(self).forward is GatedLinearRecurrence.forward and _plain(self.out)):
            return None
        if carry is None:
            carry = self.cell.initialize_carry(None, get_input_shape(inputs))
        rows, next_carry = self._gated_states(inputs, done, carry)
        return next_carry, native().dense_onto(residual, rows, self.out.weight, self.out.bias)

    def acting(self, x, norm, done, carry):
        layers = [self.cell.z, self.cell.h, self.gate]
        if not (type(self).forward is GatedLinearRecurrence.forward and _as_written(self.cell, MinGRUCell, "scan", "elements") and self.cell.fused
                and _row_layers(x, [*layers, self.out])):
            return None
        if carry is None:
            carry = self.cell.initialize_carry(None, get_input_shape(x))
        product = autocast_dtype(x) or x.dtype
        layers.append(self.out)
        y, z, *carry = native().gated_act(x, *_norm_of(norm), [m.weight for m in layers], [m.bias for m in layers], product, done, *carry,
                                          stepping_in_place())
        self.cell.intermediates.sow("gate", lambda z=z: z.float().mean())
        return tuple(carry), y

    def initialize_carry(self, key, input_shape):
        return self.cell.initialize_carry(key, input_shape)


# ----------------------------------------------------------------------------------
# acting: one time step without gradients (ppo.py:105-143), rows = environments
# ----------------------------------------------------------------------------------
_SPLIT_TERMS = 64        # the fewest terms of a sum that csrc/host_ops.cpp (SPLIT_TERMS) gives to the bfloat16 matrix units
_ACTING_ROWS = 16384   # the most rows that csrc/host_ops.cpp (rows_pay) gives to the row kernels


def _acts(x, done, norm):
    """Whether a pre-norm residual block on ``x`` is an acting step that the row kernels take."""
    return (not torch.is_grad_enabled() and x.dim() == 3 and x.shape[1] == 1 and 0 < x.shape[0] <= _ACTING_ROWS and x.is_cuda
            and x.dtype == torch.float32 and x.shape[2] % 8 == 0 and x.shape[2] <= _RMS_NORM_MAX_D and x.is_contiguous() and autocast_dtype(x) in (None, torch.bfloat16)
            and (type(norm) is _RMSNorm or (type(norm) is _LayerNorm and norm.elementwise_affine)))


def _row_layers(x, layers):
    """Whether the row kernels multiply with these layers' weights as they are (under autocast: whatever dtype the products run in), in
    less time than the array library."""
    return (all(map(_plain, layers))
            and native().row_layers_suit(x.shape[0], [m.weight for m in layers], [m.bias for m in layers], autocast_dtype(x) is not None))


def _hooked(module, deep=True):
    """Whether a hook waits in this module or (deep) below, or for every module, or an instance has a ``forward`` (``scan``, ``read``,
    ``elements``) of its own: fused operations do not run the modules they stand for."""
    return _any_global_hook() or native().any_hook(module, deep)


def _plain(layer):
    """A layer that a product with its weight stands for."""
    return type(layer) in (Dense, nn.Linear)


def _state_acts(head_dim, dtype):
    """Whether the step kernels take heads of this width as they are."""
    return head_dim <= 64 and head_dim % (16 // dtype.itemsize) == 0


def _norm_of(norm):
    """A norm as the row kernels take it: kind, scale, bias, eps."""
    if norm is None:
        return 0, None, None, 0.0
    return (1, norm.scale, None, norm.eps) if type(norm) is _RMSNorm else (2, norm.weight, norm.bias, norm.eps)


def _rows(x, norm, layers, product, out_dtype, residual=None):
    """norm(x) through the layers in one launch, as _RMSNorm / _LayerNorm / Dense would compute it; residual: added to the one result."""
    return native().row_dense(x, *_norm_of(norm), x.dtype == torch.bfloat16, [m.weight for m in layers], [m.bias for m in layers], product,
                              out_dtype, residual)


def _as_written(cell, cls, *methods):
    """A subclass that overrides what the whole-cell operations stand for (``methods``; forward, scan and read) runs its own composition."""
    return type(cell) is cls or all(getattr(type(cell), n, None) is getattr(cls, n) for n in methods or ("forward", "scan", "read"))


# ----------------------------------------------------------------------------------
# matrix-state cells
# ----------------------------------------------------------------------------------
def _norm_on_kernel(x):
    """Rows the library's norm kernels take: on the device, a multiple of four features, at most 2048."""
    return x.is_cuda and x.shape[-1] % 4 == 0 and x.shape[-1] <= _RMS_NORM_MAX_D


class _RMSNorm(nn.Module):
    """y = x * rsqrt(mean(x^2) + eps) * scale (flax.linen.RMSNorm defaults, eps = 1e-6)."""

    def __init__(self, dim, eps=1e-6):
        super().__init__()
        self.scale = nn.Parameter(torch.ones(dim))
        self.eps = eps

    def forward(self, x):
        """Statistics in float32.  On the device: the library's kernel, one pass each way, with the result in
        the dtype its readers compute in (under autocast the dense layers behind a norm would each cast it
        again); rows it does not take (wider than 2048 features, a width that is no multiple of 4) and host
        arrays go to the array library."""
        if _norm_on_kernel(x):
            return rms_norm(x, self.scale, self.eps, autocast_dtype(x) or x.dtype)
        return F.rms_norm(x.float(), (x.shape[-1],), self.scale.float(), self.eps).to(x.dtype)

    def fork(self, x):
        """(x, norm(x)) for a residual branch around this norm: with the first result used in place of x, the
        gradients of the two branches are added inside the norm's backward kernel."""
        if _norm_on_kernel(x) and x.dtype in (torch.float32, torch.bfloat16):
            return rms_norm_fork(x, self.scale, self.eps, autocast_dtype(x) or x.dtype)
        return x, self(x)


class LinearAttentionCell(MemoroidCellBase):
    """Causal linear attention with phi = elu + 1 (linear_attention.py:14-124).
    Elements are (v phi(k)^T, phi(k)) combined by addition; the reference materialises
    S (B,T,H,d,d); here the recurrence, the key sum z and the normalised read-out run in one
    chunked kernel per direction."""

    def __init__(self, features, head_dim, num_heads, in_features=None, eps=1e-6):
        super().__init__()
        in_features = features if in_features is None else in_features
        self.features, self.head_dim, self.num_heads, self.eps = features, head_dim, num_heads, eps
        hidden = head_dim * num_heads
        self.key = Dense(in_features, hidden, bias=False)
        self.value = Dense(in_features, hidden, bias=False)
        self.query = Dense(in_features, hidden, bias=False)
        self.norm = _RMSNorm(hidden)
        self.output_projection = Dense(hidden, features)

    def _heads(self, x):
        return x.view(*x.shape[:2], self.num_heads, self.head_dim)

    def forward(self, x, **kwargs):
        """Elements in kernel form: (v, k, q), keys and queries before the feature map (phi is applied
        inside the kernel).  The reference's elements are (v phi(k)^T, phi(k)); the query joins them here
        because the kernel contracts the state with it as it goes."""
        v, k, q = dense_group(x, [self.value, self.key, self.query])
        return (self._heads(v), self._heads(k), self._heads(q))

    def binary_operator(self, a, b):
        return tuple(x + y for x, y in zip(a, b))

    def scan(self, z, initial_carry, done):
        """The recurrence, the running key sum and the normalised read-out in one kernel per direction
        (the single-step kernel when T = 1 and no gradient is asked for).  Returns h = the normalised
        numerator (B,T,H,dv) and the carry (S (B,1,H,dv,dk), z (B,1,H,dk))."""
        v, k_raw, q = z
        S0, z0 = initial_carry
        out, S_last, z_last = normalised_linear_attention(q, k_raw, v, done, S0[:, 0].float(), z0[:, 0].float(),
                                                          "elu1", self.eps)
        return out, (S_last[:, None], z_last[:, None])

    def read(self, h, x, **kwargs):
        """linear_attention.py:109-117: RMS norm over the heads' concatenated outputs, then the output
        projection.  The norm is the library's kernel, one pass over the outputs each way.  (The attention
        kernels can also leave each head's sum of squares beside its outputs -- ``return_ss`` -- for a host
        that folds the rescale out * rsqrt(sum_h ss / (H d) + eps) * scale into its next operation; as array
        operations here that rescale and its gradient cost more passes than the norm kernel, which gets the
        row's statistic from the row it reads anyway: 1.72 -> 1.20 ms for this cell's forward and backward at
        1024 x 128 x 4 x 64.)"""
        layer, rows = LinearAttentionCell.closing(self, h, x)
        return layer(rows)

    def closes(self):
        return _as_written(self, LinearAttentionCell) and _plain(self.output_projection)

    def closing(self, h, x):
        return self.output_projection, self.norm(h.reshape(*x.shape[:2], -1)).to(x.dtype)

    def acting(self, x, norm, done, carry):
        layers = [self.value, self.key, self.query]
        if not (type(self.norm) is _RMSNorm and _as_written(self, LinearAttentionCell) and _row_layers(x, [*layers, self.output_projection])):
            return None
        product = autocast_dtype(x) or x.dtype
        if _state_acts(self.head_dim, product):
            layers = [self.query, self.key, self.value, self.output_projection]
            y, *carry = native().state_act(x, *_norm_of(norm), [m.weight for m in layers], [m.bias for m in layers], self.norm.scale, self.norm.eps,
                                           product, product, done, *carry, self.eps, stepping_in_place())
            return tuple(carry), y
        z = tuple(self._heads(t) for t in _rows(x, norm, layers, product, product))
        h, carry = self.scan(z, carry, done)
        return carry, _rows(h.reshape(*x.shape[:2], -1), self.norm, [self.output_projection], product, x.dtype, x)[0]

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.key.weight.device
        return (torch.zeros(*batch, 1, self.num_heads, self.head_dim, self.head_dim, device=dev),
                torch.zeros(*batch, 1, self.num_heads, self.head_dim, device=dev))


class LinearAttention(Memoroid):
    """Memoroid(LinearAttentionCell) under its own name."""

    def __init__(self, cell: LinearAttentionCell):
        super().__init__(cell)


class DeltaNetCell(MemoroidCellBase):
    """DeltaNet: S_t = S_{t-1}(I - beta_t k_t k_t^T) + beta_t v_t k_t^T, o_t = S_t q_t with
    L2-normalised keys and beta = sigmoid(.) (both formed inside the kernels).  Not in the reference; written in its cell
    idiom the elements are the affine maps (beta v k^T, I - beta k k^T) with
    binary_operator(a, b) = (B_a A_b + B_b, A_a A_b).  The carry is (S (B,1,H,d,d),)."""

    def __init__(self, features, head_dim, num_heads, in_features=None, dtype=torch.bfloat16, resets=None):
        super().__init__()
        in_features = features if in_features is None else in_features
        self.features, self.head_dim, self.num_heads, self.dtype = features, head_dim, num_heads, dtype
        self.resets = resets   # None / "passes" / "merged": mrx_reset_path, for rollouts whose episodes end often
        hidden = head_dim * num_heads
        self.query = Dense(in_features, hidden, bias=False)
        self.key = Dense(in_features, hidden, bias=False)
        self.value = Dense(in_features, hidden, bias=False)
        self.beta = Dense(in_features, num_heads, bias=False)
        self.norm = _RMSNorm(hidden)
        self.output_projection = Dense(hidden, features)

    def _heads(self, x):
        return x.view(*x.shape[:2], self.num_heads, self.head_dim)

    def forward(self, x, **kwargs):
        """The raw projections (q, k, v, beta logits): the key normalisation and the sigmoid run
        inside the kernels."""
        dt = self.dtype
        q, k, v, beta = dense_group(x, [self.query, self.key, self.value, self.beta])
        return (self._heads(q).to(dt), self._heads(k).to(dt), self._heads(v).to(dt), beta.to(dt))

    def binary_operator(self, a, b):
        B_i, A_i = a
        B_j, A_j = b
        return (B_i @ A_j + B_j, A_i @ A_j)

    def scan(self, z, initial_carry, done):
        q, k, v, beta_raw = z
        (S0,) = initial_carry
        o, S_last = deltanet(q, k, v, beta_raw, done, S0[:, 0].float(), resets=self.resets)
        return o, (S_last[:, None],)

    def read(self, h, x, **kwargs):
        layer, rows = DeltaNetCell.closing(self, h, x)
        return layer(rows)

    def closes(self):
        return _as_written(self, DeltaNetCell) and _plain(self.output_projection)

    def closing(self, h, x):
        return self.output_projection, self.norm(h.reshape(*x.shape[:2], -1)).to(x.dtype)

    def acting(self, x, norm, done, carry):
        layers = [self.query, self.key, self.value, self.beta]
        if not (type(self.norm) is _RMSNorm and _as_written(self, DeltaNetCell) and self.dtype in (torch.float32, torch.bfloat16)
                and _row_layers(x, [*layers, self.output_projection])):
            return None
        product = autocast_dtype(x) or x.dtype
        if _state_acts(self.head_dim, self.dtype):
            layers.append(self.output_projection)
            y, S, _ = native().state_act(x, *_norm_of(norm), [m.weight for m in layers], [m.bias for m in layers], self.norm.scale, self.norm.eps,
                                         product, self.dtype, done, carry[0], None, 0.0, stepping_in_place())
            return (S,), y
        q, k, v, beta = _rows(x, norm, layers, product, self.dtype)
        h, carry = self.scan((self._heads(q), self._heads(k), self._heads(v), beta), carry, done)
        return carry, _rows(h.reshape(*x.shape[:2], -1), self.norm, [self.output_projection], product, x.dtype, x)[0]

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.key.weight.device
        return (torch.zeros(*batch, 1, self.num_heads, self.head_dim, self.head_dim, device=dev),)


def _depthwise(conv):
    """A convolution that the library's causal kernel stands for: one filter a channel, with a bias, every step, nothing padded."""
    return (type(conv) is nn.Conv1d and conv.bias is not None and conv.groups == conv.in_channels == conv.out_channels
            and conv.stride == conv.dilation == (1,) and conv.padding == (0,))


def _causal_conv_silu(x, conv):
    """silu of a depthwise convolution over time that sees the steps up to its own and nothing before the call's first
    (mamba.py:88-106): the library's kernel where it takes the arrays, else the array library's operations."""
    K = conv.kernel_size[0]
    if (_depthwise(conv) and not _hooked(conv) and x.is_cuda and x.dtype == torch.float32 and conv.weight.dtype == torch.float32 and autocast_dtype(x) is None and K <= 4
            and x.shape[2] % 4 == 0 and x.numel() > 0):
        return native().causal_conv_silu(x, conv.weight, conv.bias)
    return F.silu(conv(F.pad(x.transpose(1, 2), (K - 1, 0)))).transpose(1, 2)


class MambaCell(MemoroidCellBase):
    """Mamba-2 style selective state space cell (mamba.py:33-144).  Elements are
    (h_t = (B_t dt_t) (x) x_t : (H,N,P), decay_t = exp(dt_t A) : (H,1,1)) combined by the diagonal
    operator; read is y_t = C_t . h_t + D x_t, gated by silu(z) after RMSNorm.  The reference
    materialises h (B,T,H,N,P); here the scan and the C-contraction run in the gated chunked
    kernel with k = B dt, v = x, q = C and log-decay g = dt A (native at state_dim = head_dim = 64 or
    32; other sizes are padded by the op, state_dim up to 64).
    Carry: (h (B,1,H,N,P), decay (B,1,H,1,1)), the reference's shapes."""

    def __init__(self, features, num_heads=8, head_dim=64, state_dim=64, conv_dim=4, in_features=None):
        super().__init__()
        in_features = features if in_features is None else in_features
        self.features, self.num_heads, self.head_dim = features, num_heads, head_dim
        self.state_dim, self.conv_dim = state_dim, conv_dim
        hidden, sp = num_heads * head_dim, num_heads * state_dim
        conv_channels = hidden + 2 * sp
        self.A_log = nn.Parameter(torch.empty(num_heads).uniform_(math.log(1.0), math.log(16.0)))
        self.D = nn.Parameter(torch.ones(num_heads))
        dt = torch.exp(torch.rand(num_heads) * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
        self.dt_bias = nn.Parameter(dt + torch.log(-torch.expm1(-dt)))
        self.input_projection = Dense(in_features, hidden * 2, bias=False)
        self.B = Dense(in_features, sp, bias=False)
        self.C = Dense(in_features, sp, bias=False)
        self.dt = Dense(in_features, num_heads, bias=False)
        self.conv = nn.Conv1d(conv_channels, conv_channels, conv_dim, groups=conv_channels)
        self.norm = _RMSNorm(hidden)
        self.output_projection = Dense(hidden, features)

    def _project(self, x):
        Bn, T, _ = x.shape
        H, P, N = self.num_heads, self.head_dim, self.state_dim
        up, B_in, C_in, dt_in = dense_group(x, [self.input_projection, self.B, self.C, self.dt])
        hidden, z = up.chunk(2, dim=-1)
        ci = _causal_conv_silu(torch.cat([hidden, B_in, C_in], dim=-1), self.conv)   # causal, per call
        hidden = ci[..., :H * P].reshape(Bn, T, H, P)
        B_proj = ci[..., H * P:H * P + H * N].reshape(Bn, T, H, N)
        C_proj = ci[..., H * P + H * N:].reshape(Bn, T, H, N)
        dt = F.softplus(dt_in + self.dt_bias)
        return hidden, B_proj, C_proj, z, dt

    def forward(self, x, **kwargs):
        """Elements in kernel form: (k = B dt, v = x, log-decay g = dt A, q = C); the reference's
        (h, decay) are v (x) k and exp(g), and the C projection joins them because the kernel fuses the
        contraction y_t = C_t . h_t into the scan."""
        hidden, B_proj, C_proj, _, dt = self._project(x)
        g = dt * (-torch.exp(self.A_log))[None, None, :]
        return (B_proj * dt[..., None], hidden, g, C_proj)

    def binary_operator(self, a, b):
        h_i, decay_i = a
        h_j, decay_j = b
        return (decay_j * h_i + h_j, decay_j * decay_i)

    def scan(self, z, initial_carry, done):
        k, v, g, q = z
        h0, decay0 = initial_carry                      # (B,1,H,N,P), (B,1,H,1,1)
        S0 = h0[:, 0].transpose(-1, -2).float().contiguous()   # kernel state is (P, N) = (d_v, d_k)
        o, S_last = gated_linear_attention(q.contiguous(), k.contiguous(), v.contiguous(), g.float(), done, S0)
        Bn, T, H = g.shape
        ones = torch.ones(H, device=g.device)
        _, G_last, _ = linear_scan(ones, g.float().contiguous(), done,
                                   torch.log(decay0[:, 0, :, 0, 0].float()).contiguous())
        carry = (S_last.transpose(-1, -2)[:, None], torch.exp(G_last)[:, None, :, None, None])
        return o, carry

    def whole(self, x, done, initial_carry):
        """Elements, recurrence and gated read-out in one native operation (conv_cells.hip around the gated kernels): float32
        on the device, sizes the kernels take as they are.  The composition below -- projections formed in ``forward`` and
        again in ``read``, the library's convolution between transposes -- takes ten times as long."""
        if not (self._native_sizes() and _as_written(self, MambaCell) and x.is_cuda and x.dtype == torch.float32 and x.dim() == 3 and x.shape[0] * x.shape[1] > 0 and autocast_dtype(x) is None):
            return None
        y, carry = self._mix(dense_group(x, [self.input_projection, self.B, self.C, self.dt]), done, initial_carry)
        return carry, self.output_projection(y)

    def whole_onto(self, residual, x, done, initial_carry):
        layer = self.output_projection
        if not (type(self).whole is MambaCell.whole and self._native_sizes() and _as_written(self, MambaCell) and x.is_cuda and x.dtype == torch.float32
                and x.dim() == 3 and x.shape[0] * x.shape[1] > 0 and autocast_dtype(x) is None):
            return None
        if initial_carry is None:
            initial_carry = self.initialize_carry(None, get_input_shape(x))
        y, carry = self._mix(dense_group(x, [self.input_projection, self.B, self.C, self.dt]), done, initial_carry)
        return carry, native().dense_onto(residual, y, layer.weight, layer.bias)

    def _native_sizes(self):
        P = self.head_dim
        return (type(self.norm) is _RMSNorm and self.norm.scale.dtype == torch.float32 and _plain(self.output_projection)
                and _depthwise(self.conv)
                and P % 4 == 0 and P <= 64 and self.state_dim in (4, 8, 16, 32, 64) and self.conv_dim <= 4
                and self.num_heads * P <= _RMS_NORM_MAX_D and self.conv.weight.dtype == torch.float32)

    def _mix(self, projections, done, carry):
        h0, decay0 = carry
        y, S_last, decay = native().mamba_mix(*projections, self.conv.weight, self.conv.bias, self.dt_bias, self.A_log, self.D,
                                              self.norm.scale, done, h0[:, 0].transpose(-1, -2), decay0[:, 0, :, 0, 0], self.norm.eps,
                                              stepping_in_place())
        return y, (S_last.transpose(-1, -2)[:, None], decay[:, None, :, None, None])

    def acting(self, x, norm, done, carry):
        layers = [self.input_projection, self.B, self.C, self.dt]
        if not (self._native_sizes() and _as_written(self, MambaCell) and autocast_dtype(x) is None
                and _row_layers(x, [*layers, self.output_projection])):
            return None
        y, carry = self._mix(_rows(x, norm, layers, x.dtype, x.dtype), done, carry)
        return carry, _rows(y, None, [self.output_projection], x.dtype, x.dtype, x)[0]

    def read(self, o, x, **kwargs):
        Bn, T, _ = x.shape
        hidden, _, _, z, _ = self._project(x)
        y = o.float() + self.D[None, None, :, None] * hidden
        y = y.reshape(Bn, T, self.num_heads * self.head_dim)
        return self.output_projection(_gated(self.norm(y), z).to(x.dtype))

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        dev = self.A_log.device   # (N, P) in shape, laid out as the kernels hold it: (P, N)
        return (torch.zeros(*batch, 1, self.num_heads, self.head_dim, self.state_dim, device=dev).transpose(-1, -2),
                torch.ones(*batch, 1, self.num_heads, 1, 1, device=dev))


class Mamba(Memoroid):
    """Memoroid(MambaCell) under its own name."""

    def __init__(self, cell: MambaCell):
        super().__init__(cell)


class _BlockDiagonalDense(nn.Module):
    """One dense map per head (layers/block_diagonal_dense.py:10-50), no bias."""

    def __init__(self, features, num_heads):
        super().__init__()
        bs = features // num_heads
        self.num_heads = num_heads
        self.kernel = nn.Parameter(torch.randn(num_heads, bs, bs) * math.sqrt(2.0 / (5.0 * bs)))

    def forward(self, x):
        *batch, f = x.shape
        y = torch.einsum("...hd,hod->...ho", x.reshape(*batch, self.num_heads, -1), self.kernel)
        return y.reshape(*batch, f)


class mLSTMCell(MemoroidCellBase):
    """Matrix LSTM (mlstm.py:31-240).  Elements (C = k (x) v, log_f, n = k, m = log_i) combine by the
    max-stabilised gated sum of mlstm.py:190-206; read divides q C by max(|q . n|, exp(-m)) + 1e-6.
    Unrolled, that operator is the recurrence
        m_t = max(m_{t-1} + log f_t, log i_t)
        C_t = exp(log f_t + m_{t-1} - m_t) C_{t-1} + exp(log i_t - m_t) k_t v_t^T      (n_t alike),
    a gated linear recurrence whose log-decay g_t = log f_t + m_{t-1} - m_t and key weight
    exp(log i_t - m_t) are both <= 1 whatever the gates do: m, g and the weights come from one pass per
    (b, h) in the library (functional.mlstm_gates), q C runs in the gated chunked kernel and n in the
    diagonal scan.  State, normaliser and m come out in the reference's stabilised
    units, step by step, so gates may drift by any amount inside an episode.
    Carry: (C (B,1,H,d,d), log_f (B,1,H,1,1), n (B,1,H,d,1), m (B,1,H,1,1)) as in the reference."""

    def __init__(self, features, hidden_dim, num_heads=4, conv_kernel_size=4, in_features=None):
        super().__init__()
        if hidden_dim % num_heads != 0:
            raise ValueError(f"hidden_dim ({hidden_dim}) must be divisible by num_heads ({num_heads}).")
        in_features = features if in_features is None else in_features
        self.features, self.hidden_dim, self.num_heads = features, hidden_dim, num_heads
        self.conv_kernel_size = conv_kernel_size
        self.up_projection = Dense(in_features, 2 * hidden_dim, bias=False)
        self.causal_conv = nn.Conv1d(hidden_dim, hidden_dim, conv_kernel_size, groups=hidden_dim)
        self.query = _BlockDiagonalDense(hidden_dim, num_heads)
        self.key = _BlockDiagonalDense(hidden_dim, num_heads)
        self.value = _BlockDiagonalDense(hidden_dim, num_heads)
        self.i_gate = Dense(3 * hidden_dim, num_heads)
        self.f_gate = Dense(3 * hidden_dim, num_heads)
        with torch.no_grad():
            self.i_gate.weight.zero_()
            self.i_gate.bias.normal_(std=0.1)
            self.f_gate.weight.zero_()
            self.f_gate.bias.copy_(torch.linspace(3.0, 6.0, num_heads))
        self.learnable_skip = nn.Parameter(torch.ones(hidden_dim))
        self.norm_weight = nn.Parameter(torch.zeros(num_heads, hidden_dim // num_heads))
        self.output_projection = Dense(hidden_dim, features, bias=False)

    def _project(self, x):
        Bn, T, _ = x.shape
        d = self.hidden_dim // self.num_heads
        x_mlstm, z = self.up_projection(x).chunk(2, dim=-1)
        u = _causal_conv_silu(x_mlstm, self.causal_conv)
        heads = lambda t: t.reshape(Bn, T, self.num_heads, d)  # noqa: E731
        if self._maps_native(u):
            q, k = native().head_maps(u, [self.query.kernel, self.key.kernel])
            (v,) = native().head_maps(x_mlstm, [self.value.kernel])
        else:
            q, k, v = self.query(u), self.key(u), self.value(x_mlstm)
        return heads(q), heads(k), heads(v), z, u

    def _maps_native(self, u):
        """Whether the block-diagonal maps run as one operation each way (csrc/host_ops.cpp): float32 on the device, heads of up to 64
        features, where a batched product's permutations and its weight gradients over every row cost several times its arithmetic."""
        maps = (self.query, self.key, self.value)
        return (self._few_narrow_heads(u) and u.dtype == torch.float32 and u.numel() > 0
                and all(type(m) is _BlockDiagonalDense and not _hooked(m) and m.kernel.dtype == torch.float32 for m in maps))

    def _few_narrow_heads(self, x):
        return x.is_cuda and autocast_dtype(x) is None and self.hidden_dim // self.num_heads <= 64 and self.num_heads <= 8

    def forward(self, x, **kwargs):
        """Elements in kernel form: (k / sqrt(d), v, log_i, log_f, q)."""
        return self._elements(*self._project(x)[:3])

    def _elements(self, q, k, v):
        Bn, T, H, d = q.shape
        if self._few_narrow_heads(q):   # the gates read (q | k | v) head by head: three products that add up instead of that array
            w = torch.cat([self.i_gate.weight, self.f_gate.weight]).view(2 * H, H, 3, d)
            parts = [dense(t.reshape(Bn, T, H * d), w[:, :, i].reshape(2 * H, H * d)) for i, t in enumerate((q, k, v))]
            i_pre, f_pre = (parts[0] + parts[1] + parts[2]).chunk(2, dim=-1)
            i_pre, f_pre = (t if gate.bias is None else t + gate.bias for t, gate in ((i_pre, self.i_gate), (f_pre, self.f_gate)))
        else:
            gate_input = torch.cat([q, k, v], dim=-1).reshape(Bn, T, -1)
            i_pre, f_pre = dense_group(gate_input, [self.i_gate, self.f_gate])
        log_i = i_pre.float()
        log_f = F.logsigmoid(f_pre.float())
        return (k / math.sqrt(d), v, log_i, log_f, q)

    def _parts_as_written(self):
        blocks, dense = (self.query, self.key, self.value), (self.up_projection, self.i_gate, self.f_gate, self.output_projection)
        return (all(type(m) is _BlockDiagonalDense for m in blocks) and all(map(_plain, dense)) and _depthwise(self.causal_conv)
                and self.up_projection.bias is None and self.output_projection.bias is None
                and all(m.bias is not None for m in (self.i_gate, self.f_gate)))

    def whole(self, x, done, initial_carry):
        """The composition below with the projections formed once (``read`` forms them again)."""
        if not (x.is_cuda and x.dim() == 3 and _as_written(self, mLSTMCell)):
            return None
        q, k, v, z, u = self._project(x)
        h, carry = self.scan(self._elements(q, k, v), initial_carry, done)
        return carry, self._read_out(h, x, z, u)

    def acting(self, x, norm, done, carry):
        H, d = self.num_heads, self.hidden_dim // self.num_heads
        params = [self.up_projection.weight, self.causal_conv.weight, self.causal_conv.bias, self.query.kernel, self.key.kernel, self.value.kernel,
                  self.i_gate.weight, self.i_gate.bias, self.f_gate.weight, self.f_gate.bias, self.norm_weight, self.learnable_skip,
                  self.output_projection.weight]
        if not (_as_written(self, mLSTMCell) and self._parts_as_written() and autocast_dtype(x) is None and d in (16, 32, 64) and H <= 8 and H * d <= 256
                and all(p.dtype is torch.float32 for p in params)):
            return None
        y, *carry = native().mlstm_act(x, *_norm_of(norm), params, done, list(carry), self._G_FLOOR)
        return tuple(carry), y

    def binary_operator(self, a, b):
        C_a, log_f_a, n_a, m_a = a
        C_b, log_f_b, n_b, m_b = b
        m_a_decayed = m_a + log_f_b
        m = torch.maximum(m_a_decayed, m_b)
        sa, sb = torch.exp(m_a_decayed - m), torch.exp(m_b - m)
        return (sa * C_a + sb * C_b, log_f_a + log_f_b, sa * n_a + sb * n_b, m)

    # A log-decay below this is a state multiplied by exp(-60) < 1e-26 next to a new term of weight one:
    # clamping keeps the in-chunk prefix sums of the kernel small (no cancellation between them).
    _G_FLOOR = -60.0

    def scan(self, z, initial_carry, done):
        k, v, log_i, log_f, q = z
        C0, lf0, n0, m0 = initial_carry
        Bn, T, H, d = k.shape
        ones = torch.ones(H, device=k.device)
        m0_ = m0[:, 0, :, 0, 0].float()                                          # (B,H)
        # m_t = max(m_{t-1} + log f_t, log i_t), restarted at resets; g_t = log f_t + m_{t-1} - m_t (0 at a reset:
        # it zeroes the state anyway) and the key weights exp(log i_t - m_t) <= 1: one pass per (b, h) in the library
        m, g, wk = mlstm_gates(log_i, log_f, done, m0_, self._G_FLOOR)            # each (B,T,H)
        k_in = k.float() * wk[..., None]
        S0 = C0[:, 0].float().transpose(-1, -2).contiguous()
        num, S_last = gated_linear_attention(q.float().contiguous(), k_in.contiguous(), v.float().contiguous(),
                                             g.contiguous(), done, S0)
        a = torch.exp(g)[..., None].expand(Bn, T, H, d).reshape(Bn, T, H * d).contiguous()
        nvec, n_last, _ = linear_scan(a, k_in.reshape(Bn, T, H * d).contiguous(), done,
                                      n0[:, 0, :, :, 0].float().reshape(Bn, H * d).contiguous())
        qn = (q.float() * nvec.view(Bn, T, H, d)).sum(-1)                         # (B,T,H)
        den = torch.maximum(qn.abs(), torch.exp(-m)) + 1e-6
        h_tilde = num / den[..., None]
        _, lf_last, _ = linear_scan(ones, log_f.contiguous(), done, lf0[:, 0, :, 0, 0].float().contiguous())
        carry = (S_last.transpose(-1, -2)[:, None],
                 lf_last[:, None, :, None, None],
                 n_last.view(Bn, H, d)[:, None, :, :, None],
                 m[:, -1][:, None, :, None, None])
        return h_tilde, carry

    def read(self, h_tilde, x, **kwargs):
        return self._read_out(h_tilde, x, *self._project(x)[3:])

    def _read_out(self, h_tilde, x, z, u):
        Bn, T, _ = x.shape
        y = F.layer_norm(h_tilde, (h_tilde.shape[-1],), eps=1e-5) * (1.0 + self.norm_weight)[None, None]
        y = y.reshape(Bn, T, self.hidden_dim) + self.learnable_skip * u
        return self.output_projection(_gated(y, z).to(x.dtype))

    def initialize_carry(self, key, input_shape):
        *batch, _ = input_shape
        H, d = self.num_heads, self.hidden_dim // self.num_heads
        dev = self.learnable_skip.device
        return (torch.zeros(*batch, 1, H, d, d, device=dev), torch.zeros(*batch, 1, H, 1, 1, device=dev),
                torch.zeros(*batch, 1, H, d, 1, device=dev), torch.full((*batch, 1, H, 1, 1), -1e9, device=dev))


class mLSTM(Memoroid):
    """Memoroid(mLSTMCell) under its own name."""

    def __init__(self, cell: mLSTMCell):
        super().__init__(cell)


# ----------------------------------------------------------------------------------
# block composition used by the torso configuration (blocks/{stack,residual,normalization,ffn}.py)
# ----------------------------------------------------------------------------------
class _LayerNorm(nn.LayerNorm):
    """torch.nn.LayerNorm (same parameters, same state dict) on the library's kernel where the rows fit it."""

    def forward(self, x):
        if _norm_on_kernel(x) and self.elementwise_affine:
            return layer_norm(x, self.weight, self.bias, self.eps, autocast_dtype(x) or x.dtype)
        return super().forward(x)

    def fork(self, x):
        """(x, norm(x)) for a residual branch around this norm (see _RMSNorm.fork)."""
        if _norm_on_kernel(x) and self.elementwise_affine and x.dtype in (torch.float32, torch.bfloat16):
            return layer_norm_fork(x, self.weight, self.bias, self.eps, autocast_dtype(x) or x.dtype)
        return x, self(x)


def LayerNorm(dim):
    """flax.linen.LayerNorm with its defaults: mean and variance over the last axis, eps = 1e-6,
    learned scale and bias -- the default norm of the reference's PreNorm / PostNorm."""
    return _LayerNorm(dim, eps=1e-6)


RMSNorm = _RMSNorm


class PreNorm(nn.Module):
    """normalization.py:10-35: norm, then the wrapped sequence model.  ``norm`` is a constructor taking
    the feature width (the reference's flax modules infer it); default LayerNorm as in the reference,
    ``norm=RMSNorm`` for the torso configuration."""

    def __init__(self, module, dim, norm=LayerNorm):
        super().__init__()
        self.module, self.norm = module, norm(dim)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        return self.module(self.norm(inputs), done, initial_carry, **kwargs)

    def initialize_carry(self, key, input_shape):
        return self.module.initialize_carry(key, input_shape)


class PostNorm(nn.Module):
    """normalization.py:38-65: the wrapped sequence model, then norm."""

    def __init__(self, module, dim, norm=LayerNorm):
        super().__init__()
        self.module, self.norm = module, norm(dim)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        carry, y = self.module(inputs, done, initial_carry, **kwargs)
        return carry, self.norm(y)

    def initialize_carry(self, key, input_shape):
        return self.module.initialize_carry(key, input_shape)


def _forks(block):
    """Whether ``block`` is a pre-norm block that its norm's ``fork`` and its model stand for."""
    if not (isinstance(block, PreNorm) and type(block).forward is PreNorm.forward and hasattr(block.norm, "fork")):
        return False
    norm = type(block.norm)
    return (all(getattr(norm, "fork", None) is not c.fork or norm.forward is c.forward for c in (_RMSNorm, _LayerNorm))
            and not _hooked(block, deep=False) and not _hooked(block.norm))


class Residual(nn.Module):
    """residual.py:10-30: x + module(x)."""

    def __init__(self, module):
        super().__init__()
        self.module = module

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        inner = self.module
        if (type(inner) is PreNorm and not kwargs and hasattr(inner.module, "acting") and _acts(inputs, done, inner.norm)
                and not _hooked(inner)):
            acted = inner.module.acting(inputs, inner.norm, done, initial_carry)
            if acted is not None:
                return acted
        if inputs.is_cuda and _forks(inner):   # x + f(norm(x)): one kernel takes both gradients of x
            inputs, normed = inner.norm.fork(inputs)
            if (isinstance(inner.module, SequenceModel) and not kwargs and inputs.is_cuda and inputs.dtype is torch.float32
                    and normed.dtype in (torch.bfloat16, torch.float32) and not _hooked(inner.module)):   # the closing layer adds to the stream
                summed = inner.module.onto(inputs, normed, done, initial_carry)
                if summed is not None:
                    return summed
            carry, y = inner.module(normed, done, initial_carry, **kwargs)
        else:
            carry, y = inner(inputs, done, initial_carry, **kwargs)
        if inputs.is_cuda and inputs.dtype is torch.float32 and y.dtype is torch.bfloat16:   # a mixed-precision block on a float32 stream
            return carry, native().residual_add(inputs, y)
        return carry, inputs + y

    def initialize_carry(self, key, input_shape):
        return self.module.initialize_carry(key, input_shape)


class GatedResidual(nn.Module):
    """residual.py:33-63: x + gate(Dense(x)) * module(x), the gate a dense layer of the block's width
    (with bias) on the block's input."""

    def __init__(self, module, dim, gate=torch.sigmoid):
        super().__init__()
        self.module, self.gate, self.gate_fn = module, Dense(dim, dim), gate

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        carry, y = self.module(inputs, done, initial_carry, **kwargs)
        return carry, inputs + self.gate_fn(self.gate(inputs)) * y

    def initialize_carry(self, key, input_shape):
        return self.module.initialize_carry(key, input_shape)


def gelu(x):
    """flax.linen.gelu as the reference's blocks call it (blocks/ffn.py:16,86): the tanh approximation, which is
    jax.nn.gelu's default -- not the error-function form that is the array library's."""
    return F.gelu(x, approximate="tanh")


class _Stateless(nn.Module):
    """Blocks without a recurrence (blocks/base.py:6-21): the carry is None on the way in and out."""

    def initialize_carry(self, key, input_shape):
        return None


class FFN(_Stateless):
    """ffn.py:11-50: Dense -> activation -> dropout -> Dense, hidden width features * expansion_factor."""

    def __init__(self, features, expansion_factor=4, activation=gelu, dropout_rate=0.0):
        super().__init__()
        self.up = Dense(features, features * expansion_factor)
        self.down = Dense(features * expansion_factor, features)
        self.activation, self.dropout = activation, nn.Dropout(dropout_rate)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        return None, self.down(self.dropout(self.activation(self.up(inputs))))


class Projection(_Stateless):
    """ffn.py:53-79: a single dense layer."""

    def __init__(self, in_features, features, use_bias=True):
        super().__init__()
        self.proj = Dense(in_features, features, bias=use_bias)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        return None, self.proj(inputs)


class GLU(_Stateless):
    """ffn.py:82-123: up_proj to 2 * hidden, split into (gate, value) in that order,
    activation(gate) * value, dropout, down_proj; no biases by default."""

    def __init__(self, features, expansion_factor=4, activation=gelu, dropout_rate=0.0, use_bias=False):
        super().__init__()
        hidden = features * expansion_factor
        self.up_proj = Dense(features, 2 * hidden, bias=use_bias)
        self.down_proj = Dense(hidden, features, bias=use_bias)
        self.activation, self.dropout = activation, nn.Dropout(dropout_rate)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        gate, value = self.up_proj(inputs).chunk(2, dim=-1)
        return None, self.down_proj(self.dropout(self.activation(gate) * value))


class Stack(nn.Module):
    """stack.py:10-60: one carry per block, threaded as a tuple."""

    def __init__(self, blocks):
        super().__init__()
        self.blocks = nn.ModuleList(blocks)

    def forward(self, inputs, done=None, initial_carry=None, **kwargs):
        if initial_carry is None:
            initial_carry = tuple(None for _ in self.blocks)
        x, carries = inputs, []
        for block, c in zip(self.blocks, initial_carry):
            carry, x = block(x, done=done, initial_carry=c, **kwargs)
            carries.append(carry)
        return tuple(carries), x

    def initialize_carry(self, key, input_shape):
        return tuple(b.initialize_carry(key, input_shape) if hasattr(b, "initialize_carry") else None
                     for b in self.blocks)
