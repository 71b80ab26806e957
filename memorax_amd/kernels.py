"""The kernels as functions of torch device tensors: explicit residuals, no autograd.

Every function is a call of memorax_amd._native (csrc/host_ops.cpp), which validates device / dtype /
contiguity, allocates the outputs and launches on the current HIP stream; there is no alternative code
path.
"""
from __future__ import annotations

import torch

from . import _lib

_DT = {torch.float32: _lib.MRX_F32, torch.bfloat16: _lib.MRX_BF16, torch.complex64: _lib.MRX_C64}
_FMAP = {"none": _lib.MRX_FMAP_NONE, "elu1": _lib.MRX_FMAP_ELU1}

RMS_NORM_PARTS = 1024   # MRX_RMS_NORM_PARTS: rows of the backward's workspace
RMS_NORM_MAX_D = 2048


def init(device=None):
    """Per-device set-up of the library (mrx_init): optional, the first launch on a device does
    the same, but it must precede a HIP-graph capture that holds the first call on that device."""
    lib = _lib.load()
    dev = torch.cuda.current_device() if device is None else int(device)
    _lib.check(lib.mrx_init(dev), "mrx_init")


def chunk_size(dtype, delta=False) -> int:
    """Chunk length of the (gated) linear-attention kernels, or of the delta-rule kernels."""
    return _lib.native().chunk_size(dtype, delta)


# ----------------------------------------------------------------- diagonal scan
def linear_scan_fwd(a, b, done, h0=None, P0=None, want_P=True):
    """h_t = done ? b_t : a_t h_{t-1} + b_t.  a: (B,T,D) or (D,) time-invariant.  float32, complex64, or
    bfloat16 arrays with float32 arithmetic and float32 carries (h0, P0, h_last, P_last).
    Returns (h, h_last, P_last)."""
    return _lib.native().linear_scan_fwd(a, b, done, h0, P0, want_P)


def linear_scan_bwd(a, h, done, h0, g, g_last=None, sum_da=False):
    """Returns (da (B,T,D) per step, db, dh0).  sum_da (time-invariant a only): da is (B,D), the per-step
    terms summed over the sequence inside the kernel."""
    return _lib.native().linear_scan_bwd(a, h, done, h0, g, g_last, sum_da)


def linear_scan_last(a, b, done, h0=None):
    """Final state of h_t = done ? b_t : a_t h_{t-1} + b_t with one decay per group of channels:
    a: (B,T,D/group), b: (B,T,D), h0: (B,D) or None.  Returns h_last (B,D)."""
    return _lib.native().linear_scan_last(a, b, done, h0)


def mingru_scan_fwd(z, h_tilde, done, h0=None, P0=None, want_P=True):
    """MinGRU recurrence from its two projections (min_gru.py:49-78, in linear space):
    h_t = done ? b_t : a_t h_{t-1} + b_t with a = sigmoid(-z), b = sigmoid(z) g(h~) formed inside
    the kernel.  z, h_tilde: (B,T,D) float32 or bfloat16 (float32 arithmetic); h0, P0: (B,D) float32,
    linear space.  Returns (h in the dtype of z, h_last, P_last)."""
    return _lib.native().mingru_scan_fwd(z, h_tilde, done, h0, P0, want_P)


def mingru_scan_bwd(z, h_tilde, h, done, h0, g, g_last=None):
    """Returns (dz, dh_tilde, dh0) for the states h of mingru_scan_fwd and their gradients g."""
    return _lib.native().mingru_scan_bwd(z, h_tilde, h, done, h0, g, g_last)


# ------------------------------------------------------- gates, norms, the gating product
def mlstm_gates_fwd(log_i, log_f, done, m0=None, g_floor=-60.0):
    """The mLSTM cell's stabiliser in one pass (mrx_mlstm_gates_fwd): log_i, log_f (B,T,H) float32, m0 (B,H) or
    None (the cell's initial -1e9).  Returns (m, g, w), each (B,T,H): the running maximum, the log-decay
    g_t = log_f_t + m_{t-1} - m_t (0 at a reset, not below g_floor) and the key weight exp(log_i_t - m_t)."""
    return _lib.native().mlstm_gates_fwd(log_i, log_f, done, m0, g_floor)


def mlstm_gates_bwd(log_i, log_f, done, m0, m, dm, dg, dw, g_floor=-60.0, want_dm0=True):
    """Gradients of mlstm_gates_fwd: dm, dg, dw (each (B,T,H) or None) in, (dlog_i, dlog_f, dm0) out."""
    return _lib.native().mlstm_gates_bwd(log_i, log_f, done, m0, m, dm, dg, dw, g_floor, want_dm0)


def rms_norm_fwd(x, scale, eps=1e-6, out_dtype=None):
    """y = x * rsqrt(mean(x^2) + eps) * scale over the last axis (mrx_rms_norm_fwd): x (..., D) float32 or
    bfloat16, scale (D) float32 or None (ones); y in out_dtype (default: x's)."""
    return layer_norm_fwd(x, scale, None, eps, out_dtype, center=False)


def rms_norm_bwd(x, scale, dy, eps=1e-6, want_dscale=True, dx_add=None):
    """Gradients of rms_norm_fwd: dy (..., D) float32 or bfloat16 in; (dx in x's dtype, dscale (D) float32 or
    None) out.  The statistics are recomputed from x.  dx_add (like x, or None): added to dx."""
    return layer_norm_bwd(x, scale, dy, eps, want_dscale, dx_add, center=False)[:2]


def layer_norm_fwd(x, scale, bias, eps=1e-6, out_dtype=None, center=True):
    """y = (x - mean(x)) * rsqrt(var(x) + eps) * scale + bias over the last axis (mrx_layer_norm_fwd); center=False:
    the RMS norm (no mean, no bias).  x (..., D) float32 or bfloat16; scale, bias (D) float32 or None."""
    return _lib.native().norm_fwd(x, scale, bias, eps, out_dtype, center)


def layer_norm_bwd(x, scale, dy, eps=1e-6, want_dparams=True, dx_add=None, center=True):
    """Gradients of layer_norm_fwd: (dx in x's dtype, dscale, dbias) -- the parameters' gradients (D) float32, or
    None when not wanted (dbias also None for the RMS norm).  dx_add (like x, or None): added to dx."""
    return _lib.native().norm_bwd(x, scale, dy, eps, want_dparams, dx_add, center)


def silu_gate_fwd(h, g):
    """y = h * silu(g) (mrx_silu_gate_fwd): h, g of one shape and dtype, float32 or bfloat16."""
    return _lib.native().silu_gate_fwd(h, g)


def silu_gate_bwd(h, g, dy):
    """(dh, dg) of y = h * silu(g) for the gradient dy of y."""
    return _lib.native().silu_gate_bwd(h, g, dy)


# ----------------------------------------------------------------- chunked attention
def linear_attn_chunk_parallel_pays(B, T, H, dtype):
    """The library's rule: cut the work along time (one workgroup per chunk) instead of along sequences."""
    return bool(_lib.load().mrx_linear_attn_chunk_parallel_pays(B, T, H, _DT[dtype]))


def linear_attn_fwd(q, k, v, done, S0=None, feature_map=0, save_chk=True, chunk_parallel=None):
    """Returns (o, S_last fp32, chk) with chk = (S_chk, S_last), what the backward call needs, or None.
    Sequential form (one workgroup per sequence): S_chk is float32 and sparse -- the library writes only
    the slots of chunks that contain a reset (the backward call walks the state back from S_last through
    the others).  Chunk-parallel form (chunk_parallel=True, or None and the library's rule prefers it:
    few sequences, several chunks each): S_chk is dense and chk = (S_chk, None); linear_attn_bwd takes
    either."""
    o, S_last, S_chk, parallel = _lib.native().linear_attn_fwd(q, k, v, done, S0, int(feature_map), save_chk, chunk_parallel)
    return o, S_last, ((S_chk, None if parallel else S_last) if save_chk else None)


def linear_attn_bwd(q, k, v, done, chk, do, dS_last=None, feature_map=0, want_dS0=True):
    """chk = (S_chk, S_last) from linear_attn_fwd (S_last None: the chunk-parallel pair).
    Returns (dq, dk, dv, dS0)."""
    return _lib.native().linear_attn_bwd(q, k, v, done, *chk, do, dS_last, int(feature_map), want_dS0)


def linear_attn_norm_fwd(q, k, v, done, S0=None, z0=None, feature_map=0, eps=1e-6, save_chk=True, want_ss=False):
    """Linear attention with the normalised read-out fused.
    Returns (o, den fp32 (B,H,T), S_last fp32, z_last fp32, (S_chk, z_chk, S_last) or None); S_chk as for
    linear_attn_fwd.  want_ss: a sixth result, ss fp32 (B,H,T), the per-head sums of squares of the
    outputs (what an RMS norm over the heads needs from each of them)."""
    o, den, S_last, z_last, S_chk, z_chk, ss = _lib.native().linear_attn_norm_fwd(q, k, v, done, S0, z0, int(feature_map), eps,
                                                                                 save_chk, want_ss)
    chk = (S_chk, z_chk, S_last) if save_chk else None
    return (o, den, S_last, z_last, chk, ss) if want_ss else (o, den, S_last, z_last, chk)


def linear_attn_norm_bwd(q, k, v, done, chk, o, den, do, dS_last=None, dz_last=None, feature_map=0, eps=1e-6,
                         want_d0=True, d_ss=None):
    """Returns (dq, dk, dv, dS0, dz0).  d_ss: gradient of the forward call's ss, fp32 (B,H,T)."""
    return _lib.native().linear_attn_norm_bwd(q, k, v, done, *chk, o, den, do, dS_last, dz_last, int(feature_map), eps, want_d0,
                                              d_ss)


_FACTORS = {None: _lib.MRX_FACTORS_AUTO, "auto": _lib.MRX_FACTORS_AUTO, "parallel": _lib.MRX_FACTORS_PARALLEL,
            "inline": _lib.MRX_FACTORS_INLINE}
_RESETS = {None: _lib.MRX_RESETS_AUTO, "auto": _lib.MRX_RESETS_AUTO, "passes": _lib.MRX_RESETS_PASSES,
           "merged": _lib.MRX_RESETS_MERGED}


def delta_rule_fwd_noalloc(q, k, v, beta, done, S0=None, out=None):
    """mrx_delta_rule_fwd_noalloc: forward without residuals, the triangular factors in the
    library's static scratch array (nothing is allocated by the library; this wrapper allocates
    o and S_last unless out = (o, S_last) is given).  Returns (o, S_last)."""
    return _lib.native().delta_rule_fwd_noalloc(q, k, v, beta, done, S0, *(out or (None, None)))


def delta_rule_fwd(q, k, v, beta, done, S0=None, save_chk=True, out=None, prologue=False, tm_scratch=None,
                   factor_path=None, reset_path=None):
    """Returns (o, S_last fp32, chk) where chk = (S_chk, Tm_chk) are the residuals the
    backward call needs, or None.  out = (o, S_last, S_chk, Tm_chk) reuses buffers of an earlier
    call with the same shapes instead of allocating.  prologue=True: k is L2-normalised and
    beta = sigmoid(beta) inside the kernel (mrx_deltanet_fwd).
    tm_scratch (only without residuals): give the library a buffer for the triangular factors
    anyway, which lets it compute them chunk-parallel.  None: when the library would use it (float32;
    bf16 with B*H at most two sequences per compute unit).
    factor_path: None / "auto" (by occupancy), "parallel" or "inline" (mrx_factor_path).
    reset_path: "passes" (one unit of work per episode of a chunk), "merged" (one per chunk behind a screen of its inputs, in code for
    short episodes) or None / "auto" (the library's choice: mrx_reset_path); the backward call takes the same argument."""
    if out is not None:
        save_chk = out[2] is not None
    o, S_last, S_chk, Tm_chk = _lib.native().delta_rule_fwd(q, k, v, beta, done, S0, save_chk, out, prologue, tm_scratch,
                                                            _FACTORS[factor_path], _RESETS[reset_path])
    return o, S_last, ((S_chk, Tm_chk) if save_chk else None)


def delta_rule_bwd(q, k, v, beta, done, chk, do, dS_last=None, want_dS0=True, out=None, prologue=False,
                   reset_path=None):
    """chk = (S_chk, Tm_chk) from delta_rule_fwd.  Returns (dq, dk, dv, dbeta, dS0).
    out = (dq, dk, dv, dbeta, dS0) reuses buffers instead of allocating.  prologue=True pairs with
    delta_rule_fwd(prologue=True): k and beta are the raw projections and so are dk and dbeta."""
    return _lib.native().delta_rule_bwd(q, k, v, beta, done, *chk, do, dS_last, want_dS0, out, prologue, _RESETS[reset_path])


# ---------------------------------------------------- gated linear attention
def gated_linear_attn_fwd(q, k, v, g, done, S0=None, feature_map=0, save_chk=True):
    """g: (B,T,H) float32 log-decay.  Returns (o, S_last fp32, S_chk or None)."""
    return _lib.native().gated_linear_attn_fwd(q, k, v, g, done, S0, int(feature_map), save_chk)


def gated_linear_attn_bwd(q, k, v, g, done, S_chk, do, dS_last=None, feature_map=0, want_dS0=True,
                          S_last=None):
    """Returns (dq, dk, dv, dg, dS0).  S_last (the forward call's) is needed when dS_last is given: its
    inner product with dS_last enters dg at the last step."""
    return _lib.native().gated_linear_attn_bwd(q, k, v, g, done, S_chk, do, dS_last, int(feature_map), want_dS0, S_last)


# ------------------------------------------------------------- single time step
def linear_attn_step(q, k, v, done, S=None, z=None, feature_map="none", normalise=False, eps=1e-6,
                     inplace=False):
    """One time step.  q,k,v: (B,H,d); done: (B,); S: (B,H,dv,dk) fp32 or None; z: (B,H,dk) fp32 or
    None.  Returns (o, S_new, z_new) (z_new None unless normalise).  inplace updates S and z."""
    return _lib.native().linear_attn_step(q, k, v, done, S, z, _FMAP[feature_map], normalise, eps, inplace)


def gated_linear_attn_step(q, k, v, g, done, S=None, feature_map="none", inplace=False):
    """One time step of gated linear attention.  q,k: (B,H,dk); v: (B,H,dv); g: (B,H) fp32 log-decay;
    done: (B,); S: (B,H,dv,dk) fp32 or None.  Returns (o, S_new).  inplace updates S."""
    return _lib.native().gated_linear_attn_step(q, k, v, g, done, S, _FMAP[feature_map], inplace)


def delta_rule_step(q, k, v, beta, done, S=None, inplace=False):
    """One time step of the delta rule.  beta: (B,H).  Returns (o, S_new)."""
    return _lib.native().delta_rule_step(q, k, v, beta, done, S, inplace)
