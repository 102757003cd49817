"""PyTorch operators for the two elementwise stages around the RG-LRU inside the recurrent block: the
causal depthwise convolution that feeds it (griffin/griffin.py:474-487, the all-tokens-active path)
over ``rglru_hip_conv_fwd`` / ``rglru_hip_conv_bwd``, and the output gate ``h * gelu_tanh(v)``
(griffin/griffin.py:464, :520) over ``rglru_hip_gelu_gate_fwd`` / ``_bwd`` of librglru_hip.so.

There is no CPU fallback here: the operator raises when the library or a GPU is missing.
"""

from __future__ import annotations

from functools import lru_cache

import torch
from torch import Tensor

from . import _lib
# _ptr and _stream_ptr: for callers that drive the C ABI directly
from .hip_scan import FIRST_TOKEN_RESET, _DTYPE_CODES, _dtype_code, _ptr, _stream_ptr


@lru_cache(maxsize=None)
def max_kernel_size() -> int:
    """Largest convolution kernel size the HIP kernels cover."""
    return int(_lib.load().rglru_hip_conv_max_kernel_size())


def hip_causal_conv(u: Tensor, state: Tensor | None, weight: Tensor, bias: Tensor | None,
                    segment_pos: Tensor, need_state: bool = True) -> tuple[Tensor, Tensor | None]:
    """Depthwise causal convolution with per-document tap masking.

    ``u`` [B, T, W]; ``state`` [B, K-1, W] or None (zeros); ``weight`` [W, 1, K] and ``bias`` [W] of a
    depthwise ``nn.Conv1d``; ``segment_pos`` [B, T] integer positions (a tap reaching back ``lag`` tokens
    contributes only where ``segment_pos >= lag``).  Returns ``(out [B, T, W], new_state [B, K-1, W])``;
    ``new_state`` is the last K-1 rows of ``cat(state, u)`` (griffin/griffin.py:487), or None when the
    caller says it does not need it (a training step that returns no cache).
    """
    out = _lib.native().causal_conv(u, state, weight, bias, segment_pos)
    if not need_state:
        return out, None
    history = weight.size(2) - 1
    steps = u.size(1)
    if steps >= history:
        new_state = u[:, steps - history:].clone()
    else:
        previous = u.new_zeros(u.size(0), history, u.size(2)) if state is None else state.to(u.dtype)
        new_state = torch.cat((previous[:, steps:], u), dim=1)
    return out, new_state


def hip_causal_conv_padded(u: Tensor, state: Tensor | None, weight: Tensor, bias: Tensor | None,
                           segment_pos: Tensor, active_mask: Tensor) -> tuple[Tensor, Tensor]:
    """The convolution over right-padded batches (griffin/griffin.py:488-510): inactive tokens give zeros
    and stay out of the window of previous inputs, an active token at position 0 clears the window.
    Returns ``(out [B, T, W], new_state [B, K-1, W])``.  ``out`` is differentiable in ``u``, ``state``,
    ``weight`` and ``bias``; ``new_state`` (the cache handed to the next call) carries no gradient."""
    return _lib.native().causal_conv_padded(u, state, weight, bias, segment_pos, active_mask)


def hip_gelu_gate(h: Tensor, v: Tensor) -> Tensor:
    """``h * gelu(v, approximate="tanh")`` in one pass, differentiable in both arguments."""
    return _lib.native().gelu_gate(h, v)


@lru_cache(maxsize=None)
def hip_block_forward_covers(width: int, blocks: int, taps_count: int, dtype: torch.dtype) -> bool:
    """Whether ``hip_block_forward`` has a kernel for this shape (rglru_hip_block_fwd_path)."""
    if dtype not in _DTYPE_CODES or blocks <= 0 or width % blocks:
        return False
    return bool(_lib.load().rglru_hip_block_fwd_path(width, blocks, taps_count, _DTYPE_CODES[dtype]))


def hip_block_flags(segment_pos: Tensor) -> Tensor:
    """Per-token flag bytes of ``hip_block_forward`` for integer positions [B, T] (rglru_hip_block_flags):
    reset where a document starts (position 0) and, in bits 2-3, how many convolution lags reach in front
    of the token's document."""
    return _lib.native().block_flags(segment_pos)


def hip_block_forward(u: Tensor, v: Tensor, conv_state: Tensor | None, weight: Tensor, bias: Tensor | None,
                      segment_pos: Tensor, flags: Tensor | None, w_a: Tensor, b_a: Tensor, w_x: Tensor, b_x: Tensor,
                      lam: Tensor, h0: Tensor | None, c: float = 8.0, prep=None, rows: Tensor | None = None, need_state: bool = True, around=None):
    """``gelu_tanh(v) * RG_LRU(conv(u))`` for whole sequences with every token active, one forward launch.

    ``u``, ``v`` [B, T, W]: the block's two projections; ``conv_state`` [B, K-1, W] or None; ``weight``
    [W, 1, K], ``bias`` [W] of the depthwise ``nn.Conv1d`` (K <= 4); ``segment_pos`` [B, T]; ``flags``:
    ``hip_block_flags(segment_pos)`` if the caller has it already, ``hip_scan.FIRST_TOKEN_RESET`` when the
    positions are 0 .. T-1 in every row (no flag tensor is needed then), else None; the five RG-LRU parameters, ``h0`` [B, W] or None; ``prep``: a prepared parameter image to use
    when no gradient is asked for.  For right-padded batches ``rows``, ``segment_pos`` and ``flags`` are the rows,
    conv_positions and flags of ``token_facts``; the new convolution state then carries no gradient and is computed only
    if ``need_state``.  Returns ``(gated [B, T, W], final state [B, W] fp32, new_conv_state
    [B, K-1, W])``; differentiable in u, v, the parameters, conv_state and h0.

    ``around``: (x [B, T, D], the weights and biases of linear_x, linear_y and linear_out, activity mask or None) puts the Linear
    layers into the operator: the whole block of a training step without cache, one node of the graph.  u and v are then None,
    or the projections of x if the caller has them already (``hip_linear_pair_values``).  Returns ``(output [B, T, D], None,
    None)``; the output is None where the node does not take the operands (the caller then goes layer by layer).
    """
    first_reset = flags is FIRST_TOKEN_RESET
    if around is not None:
        x, w_u, b_u, w_v, b_v, w_o, b_o, active = around
        return _lib.native().block_train(x, (w_u, b_u, w_v, b_v, weight, bias, w_a, b_a, w_x, b_x, lam, w_o, b_o), segment_pos,
                                         None if first_reset else flags, rows, active, u, v, first_reset, c), None, None
    gated, h_last, new_conv = _lib.native().block_forward(
        u, v, conv_state, weight, bias, segment_pos, None if first_reset else flags, first_reset, w_a, b_a, w_x, b_x, lam, h0,
        c, None if prep is None else prep.image, rows, need_state)
    if rows is None and torch.is_grad_enabled() and (u.requires_grad or (conv_state is not None and conv_state.requires_grad)):
        # the carried rows as a differentiable function of u and conv_state (the kernel's copy carries no gradient)
        history, steps = weight.size(2) - 1, u.size(1)
        if steps >= history:
            new_conv = u[:, steps - history:].clone()
        else:
            previous = u.new_zeros(u.size(0), history, u.size(2)) if conv_state is None else conv_state.to(u.dtype)
            new_conv = torch.cat((previous[:, steps:], u), dim=1)
    return gated, h_last, new_conv


def hip_block_may_pack(x: Tensor, w: Tensor) -> bool:
    """Whether a right-padded batch ``x`` [B, T, D] trains without its padding (``hip_block_train_packed``) if there is enough of it."""
    return _lib.native().block_may_pack(x, w)


def hip_block_projections(x: Tensor, w_u: Tensor, b_u: Tensor | None, w_v: Tensor, b_v: Tensor | None):
    """The values of linear_x and linear_y for ``hip_block_train_packed``; the second is None where it would be a launch of its own and is
    better made for the active tokens alone."""
    return _lib.native().block_projections(x, w_u, b_u, w_v, b_v)


def hip_block_train_packed(x: Tensor, parameters, facts, u: Tensor, v: Tensor | None, c: float) -> Tensor | None:
    """``hip_block_forward`` with ``around`` on a batch whose rows are right-padded documents from their beginning: products and scans
    run on the active tokens alone, packed one row behind the other.  ``facts``: resolved ``token_facts`` of the mask; ``u``, ``v``:
    ``hip_block_projections``.  Returns the output [B, T, D], or None where there is too little padding, or the operator does not
    take the operands."""
    native = _lib.native()
    rows = native.block_packed_rows(x.shape[0], x.shape[1], facts.active_tokens)
    if rows == 0:
        return None
    return native.block_train_packed(x, parameters, facts.conv_positions, facts.rows, u, v, rows, c)


def hip_block_decode_step(u: Tensor, v: Tensor, conv_state: Tensor | None, weight: Tensor, bias: Tensor | None,
                          prev_pos: Tensor | None, segment_pos: Tensor | None, active: Tensor | None,
                          prep, rnn_state: Tensor | None):
    """One token per row through conv -> RG-LRU step -> output gate (no autograd), two kernel launches.

    ``u``, ``v`` [B, W]: the block's two projections of the token (rows may be strided views of one wider
    buffer); ``conv_state`` [B, K-1, W] or None;
    ``prev_pos`` [B] (None: -1) or explicit ``segment_pos`` [B]; ``active`` [B] uint8 or None (all
    active); ``prep`` the prepared RG-LRU parameters; ``rnn_state`` [B, W] fp32 or None (zeros).
    Returns ``(gated [B, W], new_rnn_state, new_conv_state, new_pos)``; the inputs are left untouched.
    """
    return _lib.native().block_decode_step(u, v, conv_state, weight, bias, prev_pos, segment_pos, active, prep.image,
                                           prep.width, prep.blocks, prep.dtype, rnn_state)


def hip_block_step(x: Tensor, linear_x, linear_y, conv, linear_out, conv_state: Tensor | None, prev_pos: Tensor | None,
                   segment_pos: Tensor | None, active: Tensor | None, prep, rnn_state: Tensor | None):
    """The block on one token per row, ``x`` [B, 1, D] (no autograd), in three launches: both projections with positions and
    convolution, the RG-LRU step with the output gate, the output projection.  The four layers are those of the block, the
    other arguments as for ``hip_block_decode_step``.  Returns ``(output [B, 1, D], rnn_state, conv_state, positions)``,
    or None where the kernels do not take the operands."""
    # nn.Module's attribute lookup costs half a microsecond a name
    px, py, pc, po = linear_x._parameters, linear_y._parameters, conv._parameters, linear_out._parameters
    try:
        operands = (px["weight"], px["bias"], py["weight"], py["bias"], pc["weight"], pc["bias"], po["weight"], po["bias"])
    except KeyError:                                         # a parametrised or otherwise replaced parameter
        operands = (linear_x.weight, linear_x.bias, linear_y.weight, linear_y.bias, conv.weight, conv.bias, linear_out.weight,
                    linear_out.bias)
    return _lib.native().block_step(x, *operands, conv_state, prev_pos, segment_pos, active, prep.image, prep.blocks, rnn_state)


def hip_block_step_captured(batch: int, width: int, dim: int) -> bool:
    """Whether ``hip_block_step`` takes so many rows inside a graph capture, where the line to the BLAS library's products lies
    lower than outside (host time is nothing in a graph)."""
    return _lib.native().own_projections_captured(3.0 * batch * width * dim)


def hip_block_infer(x: Tensor, parameters, prep, conv_state: Tensor | None, rnn_state: Tensor | None, prev_pos: Tensor | None,
                    segment_pos: Tensor | None, flags: Tensor | None, rows: Tensor | None, active: Tensor | None, u: Tensor | None,
                    v: Tensor | None, need_state: bool):
    """The whole recurrent block over sequences without gradients (griffin/griffin.py:459-528), three launches (four behind the BLAS library's products).  ``parameters``:
    weights and biases of linear_x, linear_y and the convolution, the five of the RG-LRU, weight and bias of linear_out; ``prep`` the
    image of the RG-LRU's.  Every token active: positions follow ``prev_pos`` [B] or are ``segment_pos`` [B, T].  Right-padded:
    ``flags`` and ``rows`` of ``token_facts``, ``active`` the mask.  ``u``, ``v``: the projections if the caller has them.  Returns
    ``(output, final state, convolution state, last position or None)``, or None where the kernels do not take the operands."""
    return _lib.native().block_infer(x, parameters, prep.image, conv_state, rnn_state, prev_pos, segment_pos, flags, rows, active, u, v,
                                     need_state)


def _sum_sets(sets: Tensor) -> Tensor:
    """``sets.sum(0)`` for a contiguous [sets, ...] tensor on the GPU by a kernel of the library (one pass over the
    sets, 16-byte accesses; the generic reduction takes about three times as long for eight sets of a weight
    gradient); anything else goes to ``sum``."""
    return _lib.native().sum_sets(sets)


def _stacked_halves(a: Tensor | None, b: Tensor | None) -> Tensor | None:
    """The [rows, 2 W] matrix whose column halves ``a`` and ``b`` ([..., W] each) are, or None if they are not
    laid out that way (same storage, b starts W elements behind a, rows 2 W elements apart)."""
    if a is None or b is None:
        return None
    return _lib.native().stacked_halves(a, b)


def hip_linear(x: Tensor, weight: Tensor, bias: Tensor | None, active: Tensor | None = None) -> Tensor:
    """``x @ weight.T + bias`` (griffin/griffin.py:379-389, the block's Linear layers) with the bias
    gradient reduced by a kernel of this library; differentiable in all three arguments.  ``active`` [...]: a mask of
    the rows; those where it is False come out as zeros (griffin/griffin.py:522-523)."""
    return _lib.native().linear(x, weight, bias, active)


def token_facts(active_mask: Tensor, segment_pos: Tensor | None, previous_position: Tensor | None):
    """What an activity mask [B, T] says about every token, in one launch: an object with ``positions`` [B, T] (given, or
    previous + running count of active tokens), ``flags`` / ``conv_positions`` / ``rows`` for ``hip_block_forward``,
    ``last_position`` [B], and ``resolve() -> (every token is active, every row is right-padded)``, which waits for that
    launch but not for work queued behind it."""
    return _lib.native().TokenFacts(active_mask, segment_pos, previous_position)


def hip_linear_pair(x: Tensor, w1: Tensor, b1: Tensor | None, w2: Tensor, b2: Tensor | None,
                    values: tuple[Tensor, Tensor] | None = None) -> tuple[Tensor, Tensor]:
    """``(x @ w1.T + b1, x @ w2.T + b2)``: two ``hip_linear`` calls whose backward passes share the input
    gradient (the second GEMM accumulates into the first one's result).  ``values``: the two results of
    ``hip_linear_pair_values`` on the same operands, which then only get their graph."""
    u, v = (None, None) if values is None else values
    return _lib.native().linear_pair(x, w1, b1, w2, b2, u, v)


def hip_linear_pair_values(x: Tensor, w1: Tensor, b1: Tensor | None, w2: Tensor, b2: Tensor | None) -> tuple[Tensor, Tensor]:
    """The values of ``hip_linear_pair`` without a graph behind them."""
    return _lib.native().linear_pair_values(x, w1, b1, w2, b2)


def hip_linear_values(x: Tensor, w: Tensor, b: Tensor | None) -> Tensor:
    """The value of ``hip_linear`` without a graph behind it."""
    return _lib.native().linear_values(x, w, b)


@lru_cache(maxsize=None)
def rmsnorm_max_width(dtype: torch.dtype, aligned: bool = True) -> int:
    return int(_lib.load().rglru_hip_rmsnorm_max_width(_dtype_code(dtype), 1 if aligned else 0))


def hip_rmsnorm(x: Tensor, g: Tensor, eps: float = 1e-6) -> Tensor:
    """``x * rsqrt(mean(x^2, -1) + eps) * (1 + g)`` (griffin/griffin.py:68-80), differentiable in x and g."""
    return _lib.native().rmsnorm(x, g, eps)
