"""Autograd operator of the ring-attractor time loop, HIP-backed.

Same public names, argument order and semantics as the reference's cpp/ring_rnn_cuda.py:18-144:
`ring_rnn_cuda_func(action_signal, Wa, J0, J1, Wo, r_init, alpha, activation='relu')` returns
bump_history [T,B,N] and is differentiable w.r.t. Wa and Wo.  A star-import also hands out `torch`,
which the reference training script relies on (train_general_ring_no_gain.py:19, 40).
"""
from os import environ as _environ

import torch
from torch.autograd import Function

from . import _lib
from .rnn_cuda import fwd_cuda, bwd_cuda, saved_nbytes

_ACTIVATION_MAP = {'relu': 0, 'gelu': 1, 'tanh': 2, 'silu': 3}   # cpp/ring_rnn_cuda.py:63


def _activation_id(name):
    if name not in _ACTIVATION_MAP:
        raise ValueError(f"Invalid activation '{name}'. Must be one of {list(_ACTIVATION_MAP.keys())}.")
    return _ACTIVATION_MAP[name]


def ring_rnn_cuda_func(action_signal, Wa, J0, J1, Wo, r_init, alpha, activation='relu', driven_channels=None,
                       precise_wo=None):
    """Ring RNN forward pass on the GPU.

    action_signal (B,T,k); Wa (k,N,N); J0, J1 scalars; Wo (N,N); r_init (B,N); alpha float;
    activation in {'relu','gelu','tanh','silu'}.  Returns bump_history (T,B,N).

    driven_channels (optional, not in the reference): the caller's statement that every action channel outside this
    list of at most two indices is identically zero (the training script's zero padding of (L, R) to a_dim = 16);
    see `_driven_pair`.  Tensors made by `host.av_to_action_signal_ND(zero_padding=True)` carry it themselves.

    precise_wo (optional, not in the reference; None takes the module's PRECISE_WO): Wo enters the contraction as
    two bf16 operands, its bf16 rounding and the rounding of what that leaves; see `_split_wo`.
    """
    pair = None
    if PRECISE_WO if precise_wo is None else precise_wo:
        action_signal, Wa = _split_wo(action_signal, Wa, J1, Wo)
    else:
        pair = _driven_pair(action_signal, Wa, driven_channels)
    # Autograd switches gradient mode off inside Function.forward, and needs_input_grad stays True under
    # torch.no_grad(): the wrapper is the place that knows whether a backward can follow.
    return RingRnnCudaFunc.apply(action_signal, Wa, J0, J1, Wo, r_init, alpha, activation, torch.is_grad_enabled(), pair)


# Store or recompute.  False (default): a forward that a backward can follow also writes the derivative record and the
# bf16 operand copy (ringattr_saved_bytes: 4 bytes per state element and step) for the backward to read.  True: the
# forward writes only bump_history, as the reference's does (cpp/ring_rnn_cuda.py:68-78), and the backward recomputes
# both from it before the reverse-time loop (the reference recomputes re in every backward,
# cpp/kernels/bwd_mixed_precision_aggressive.cuh:53-269): no saved buffer is held between forward and backward.
RECOMPUTE_IN_BACKWARD = False

# Default of ring_rnn_cuda_func's precise_wo.
PRECISE_WO = False


def _split_wo(action_signal, Wa, J1, Wo):
    """Wo as two bf16 MFMA operands.  The kernels round every weight to bf16 once, which makes the network they
    simulate a fixed perturbation (2^-9 relative per weight) of the caller's.  Where the dynamics are marginally
    stable -- the integrator regime the ring attractor is trained for, J1 = 1 with weights ~ N(0, 1/N) -- the two
    networks' states drift apart linearly in time: at N = 512, J0 = -1/N, J1 = 1, tanh the per-step deviation from
    fp64 reaches 1e-2 at t = 166 and 1.2e-1 at t = 511, all of it from the rounding of Wo (Wa is gated by |av| <=
    0.31 and the state operand's rounding does not accumulate; the reference's own tensor-core path keeps Wo in fp32
    and rounds Wa and the action signal, cpp/kernels/fwd_1loop_tc_idx.cuh:6-48).  With Wo = hi + lo, hi = bf16(Wo)
    and lo = bf16(Wo - hi), the deviation stays under 4e-3 over the 512 steps.
    lo rides as one more action matrix whose gate is the constant J1, so the kernels need no change: one more
    matrix in the step's weight stream (a third more work at two action channels; with N <= 256 the call moves
    from the weight-resident kernels to the streaming ones, whose matrix count is free).  The extra channel's weight
    gradient repeats grad_Wo and is dropped; gradients of Wa, Wo and, if asked for, action_signal are unchanged in
    meaning."""
    B, T, k = action_signal.shape
    lo = (Wo - Wo.to(torch.bfloat16).to(Wo.dtype)).detach()
    Wa_ext = torch.cat([Wa, lo.unsqueeze(0)], dim=0)
    gate = torch.full((B, T, 1), float(J1), dtype=action_signal.dtype, device=action_signal.device)
    return torch.cat([action_signal, gate], dim=2), Wa_ext


DRIVEN_ATTR = "_ring_driven_channels"     # set on zero-padded action signals by the host helper that builds them


def _driven_pair(action_signal, Wa, driven_channels=None):
    """The training script pads the two driven action channels with zeros up to a_dim = 16
    (train_general_ring_no_gain.py:52-66 of the reference).  A channel that is zero for every sample and step
    contributes nothing forward and has an exactly zero weight gradient, so when the caller states which (at most
    two) channels are driven and N fits the weight-resident kernels (128 < N <= 256), the operator runs on those two
    (`_compact`); silent channels get exactly zero gradients.  Returns their indices, or None for the operator on all channels.

    Nothing here reads the device back: which channels are driven comes from the caller (`driven_channels=`, or the
    attribute the host helper leaves on the tensors it pads), so the call stays asynchronous and capturable.  The
    statement is checked on the device: if a channel declared silent is not, the compacted action signal is
    poisoned with NaN, which the kernels carry into every output instead of returning a plausible wrong result.
    At other widths fewer matrices cost less too (us per pass with 16 channels and with the two: N = 800, B = 100, T = 120,
    forward and backward 8116 and 700; N = 512, B = 512, T = 120 2146 and 615), but a padded tensor that has been written to
    since must give its own results there, and its version counter does not see every write (`.data`, DLPack, a kernel
    that has its address).
    Without a statement the operator runs on all channels (the general kernels skip all-zero channels step by step).
    RINGATTR_COMPACT_CHANNELS=0 switches the compaction off."""
    if _environ.get("RINGATTR_COMPACT_CHANNELS", "1") == "0":
        return None
    if driven_channels is None:
        driven_channels = getattr(action_signal, DRIVEN_ATTR, None)
    if driven_channels is None:
        return None
    if action_signal.dim() != 3 or Wa.dim() != 3 or not action_signal.is_cuda:
        return None
    k, N = action_signal.shape[2], Wa.shape[1]
    if k <= 2 or not (128 < N <= 256) or Wa.shape[0] != k:
        return None
    if action_signal.requires_grad:        # dL/dA of a silent channel is not zero: keep every channel
        return None
    driven = sorted(set(int(c) for c in driven_channels))
    if len(driven) > 2 or any(c < 0 or c >= k for c in driven):
        raise ValueError(f"driven_channels must name at most two channels in [0, {k}), got {list(driven_channels)}")
    # (what the operator refuses, it refuses in the call on all channels)
    if action_signal.dtype != torch.float32 or Wa.dtype != torch.float32 or Wa.device != action_signal.device \
            or Wa.shape[2] != N or action_signal.numel() == 0:
        return None
    for c in range(k):                     # fewer than two driven: fill up with silent ones (their gates are zero)
        if len(driven) == 2:
            break
        if c not in driven:
            driven.append(c)
    return tuple(sorted(driven))


def _compact(action_signal, Wa, pair):
    """The two named channels' signal [B,T,2] and matrices [2,N,N]; the signal is NaN if another channel is driven."""
    B, T, k = action_signal.shape
    N = Wa.shape[1]
    dev = action_signal.device
    lib = _lib.load()
    with _lib.on_device(dev):
        a2 = torch.empty(B, T, 2, dtype=torch.float32, device=dev)
        Wa2 = torch.empty(2, N, N, dtype=torch.float32, device=dev)
        nbytes = lib.ringattr_compact_workspace_bytes()
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        _lib.check(lib.ringattr_compact_channels(action_signal.data_ptr(), Wa.data_ptr(), a2.data_ptr(), Wa2.data_ptr(), N, k, T, B,
                                                 pair[0], pair[1], ws.data_ptr(), nbytes,
                                                 _lib.stream_handle(dev)))
    return a2, Wa2


def _grad_buffers(Wa, full_shape, pair):
    """(dL/dWa, the part of it that the backward writes): all of it, or the two driven channels of a zeroed whole."""
    if pair is None:
        grad = torch.empty_like(Wa)
        return grad, grad
    grad = torch.zeros(full_shape, device=Wa.device, dtype=Wa.dtype)
    part = grad[pair[0]:pair[0] + 2]
    if pair[1] != pair[0] + 1 or part.data_ptr() % 16:
        part = torch.empty_like(Wa)
    return grad, part


def _grad_gather(grad, part, pair):
    if pair is not None and part.data_ptr() != grad[pair[0]].data_ptr():
        grad[pair[0]] = part[0]
        grad[pair[1]] = part[1]
    return grad


class RingRnnCudaFunc(Function):
    @staticmethod
    def forward(ctx, action_signal, Wa, J0, J1, Wo, r_init, alpha, activation_name, grad_mode=None, pair=None):
        activation_type = _activation_id(activation_name)
        batch_size, seq_len, a_dim = action_signal.shape
        N = Wa.shape[1]
        action_signal = action_signal.contiguous()
        Wa_c, Wo_c, r0 = Wa.contiguous(), Wo.contiguous(), r_init.contiguous()
        ctx.pair, ctx.Wa_shape = pair, Wa.shape
        if pair is not None:
            action_signal, Wa_c = _compact(action_signal, Wa_c, pair)
            a_dim = 2
        bump_history = torch.empty(seq_len, batch_size, N, device=action_signal.device, dtype=action_signal.dtype)

        # F'(re) and the bf16 operand copy of r_prev are only worth writing when a backward will follow
        # (grad_mode is None when apply() is called with the reference's eight arguments)
        needs_grad = grad_mode is not False and any(ctx.needs_input_grad[i] for i in (0, 1, 4, 5))
        ctx.extra_inputs = 0 if grad_mode is None else 2
        saved = None
        if needs_grad and not RECOMPUTE_IN_BACKWARD:
            saved = torch.empty(saved_nbytes(N, a_dim, seq_len, batch_size), dtype=torch.uint8,
                                device=action_signal.device)
        fwd_cuda.fwd(A=action_signal, Wa=Wa_c, J0=J0, J1=J1, Wo=Wo_c, r_init=r0, bump_history=bump_history,
                     alpha=alpha, activation_type=activation_type, saved=saved)

        ctx.save_for_backward(action_signal, Wa_c, Wo_c, bump_history, r0, saved)
        ctx.J0, ctx.J1, ctx.alpha, ctx.activation_type = J0, J1, alpha, activation_type
        return bump_history

    @staticmethod
    def backward(ctx, grad_output):
        action_signal, Wa, Wo, bump_history, r_init, saved = ctx.saved_tensors
        # written, not accumulated into: no zero-fill launches (but for silent channels)
        grad_Wa, part = _grad_buffers(Wa, ctx.Wa_shape, ctx.pair)
        grad_Wo = torch.empty_like(Wo)
        # The reference returns None for action_signal and r_init (cpp/ring_rnn_cuda.py:144); here they get their
        # gradients when the caller asked for them (gain networks in front of the op need dL/d action_signal).
        grad_A = torch.empty_like(action_signal) if ctx.needs_input_grad[0] else None
        grad_r0 = torch.empty_like(r_init) if ctx.needs_input_grad[5] else None
        bwd_cuda.bwd(grad_output=grad_output.contiguous(), A=action_signal, Wa=Wa, J0=ctx.J0, J1=ctx.J1, Wo=Wo,
                     bump_history=bump_history, r_init=r_init, grad_Wa=part, grad_Wo=grad_Wo,
                     alpha=ctx.alpha, activation_type=ctx.activation_type, saved=saved, grad_A=grad_A,
                     grad_r_init=grad_r0, accumulate=False)
        return (grad_A, _grad_gather(grad_Wa, part, ctx.pair), None, None, grad_Wo, grad_r0, None, None) + (None,) * ctx.extra_inputs
