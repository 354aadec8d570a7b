"""Gain networks of the action signal as one HIP operator (forward and backward).

`ring_gain_func(base_signal, params)` evaluates, per channel c, the reference models' gain network
nn.Sequential(Linear(1,h), GELU, Linear(h,1), Softplus) on |x| and returns x * gain (train/train_ring_attractor.py:70-79,
136-146; train/train_general_ring_attractor.py:38-46, 99-109).  `params` is [k, 3h+1] = per channel [w1 | b1 | w2 | b2];
`pack_gain_nets` builds it from the nn.Sequential modules with differentiable torch ops, so autograd carries the
operator's parameter gradients back into the modules.  `ring_gain_nets` and `ring_gain_halves` take the modules: the kernels
then read the parameters where they are, and their gradients are slices of one buffer.
"""
from __future__ import annotations

import ctypes

import torch
from torch.autograd import Function

from . import _lib


def pack_gain_nets(nets):
    """[k, 3h+1] parameter block of a list of nn.Sequential(Linear(1,h), GELU, Linear(h,1), Softplus)."""
    rows = []
    for net in nets:
        lin1, lin2 = net[0], net[2]
        rows.append(torch.cat([lin1.weight.reshape(-1), lin1.bias.reshape(-1), lin2.weight.reshape(-1),
                               lin2.bias.reshape(-1)]))
    return torch.stack(rows)


def _check(name, t, shape):
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a GPU tensor (device {t.device}); there is no CPU path")
    if t.dtype != torch.float32:
        raise TypeError(f"{name} must be float32, got {t.dtype}")
    if tuple(t.shape) != tuple(shape):
        raise ValueError(f"{name} must have shape {tuple(shape)}, got {tuple(t.shape)}")


class RingGainFunc(Function):
    @staticmethod
    def forward(ctx, base_signal, params):
        if base_signal.dim() != 3:
            raise ValueError(f"base_signal must be [batch, seq_len, a_dim], got {tuple(base_signal.shape)}")
        B, T, k = base_signal.shape
        if params.dim() != 2 or params.shape[0] != k or (params.shape[1] - 1) % 3 != 0:
            raise ValueError(f"params must be [a_dim, 3*hidden+1] with a_dim = {k}, got {tuple(params.shape)}")
        h = (params.shape[1] - 1) // 3
        x, prm = base_signal.contiguous(), params.contiguous()
        _check("base_signal", x, (B, T, k))
        _check("params", prm, (k, 3 * h + 1))
        lib = _lib.load()
        out = torch.empty_like(x)
        with _lib.on_device(x.device):
            _lib.check(lib.ringattr_gain_fwd(x.data_ptr(), prm.data_ptr(), out.data_ptr(), k, h, T, B,
                                             _lib.stream_handle(x.device)))
        ctx.save_for_backward(x, prm)
        ctx.dims = (B, T, k, h)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x, prm = ctx.saved_tensors
        B, T, k, h = ctx.dims
        lib = _lib.load()
        g = grad_out.contiguous()
        grad_prm = torch.empty_like(prm)
        grad_x = torch.empty_like(x) if ctx.needs_input_grad[0] else None
        with _lib.on_device(x.device):
            nbytes = lib.ringattr_gain_workspace_bytes(k, h, T, B)
            if nbytes == 0:
                _lib.check(1)
            ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
            _lib.check(lib.ringattr_gain_bwd(x.data_ptr(), prm.data_ptr(), g.data_ptr(), grad_prm.data_ptr(),
                                             grad_x.data_ptr() if grad_x is not None else None, k, h, T, B,
                                             ws.data_ptr(), nbytes, _lib.stream_handle(x.device)))
        return grad_x, grad_prm


def ring_gain_func(base_signal, params):
    """[B,T,k] base signal, [k,3h+1] packed gain-network parameters -> [B,T,k] gated action signal."""
    return RingGainFunc.apply(base_signal, params)


class RingGainNetsFunc(Function):
    """The same operator with the modules' own parameter tensors (four per channel) as inputs, for a signal that needs no
    gradient; halves: the signal is an angular velocity [B,T] and the channels are relu(-av) and relu(av).  The forward kernel
    leaves a copy of the parameters, and of an angular velocity, for the backward: either may be written to in between, as
    where `pack_gain_nets` and the two halves make new tensors."""

    @staticmethod
    def forward(ctx, signal, halves, *params):
        B, T = signal.shape[:2]
        k, h = len(params) // 4, params[0].numel()
        ctx.dims = (B, T, k, h, halves)
        out = torch.empty(B, T, k, dtype=signal.dtype, device=signal.device)
        kept = None
        if any(ctx.needs_input_grad):
            kept = torch.empty(k * (3 * h + 1) + (B * T if halves else 0), dtype=signal.dtype, device=signal.device)
            ctx.save_for_backward(kept, None if halves else signal)
        with _lib.on_device(signal.device):
            _lib.check(_lib.load().ringattr_gain_nets_fwd_kept(signal.data_ptr(), int(halves), _pointers([p.data_ptr() for p in params]),
                                                               out.data_ptr(), kept.data_ptr() if kept is not None else None, k, h, T, B,
                                                               _lib.stream_handle(signal.device)))
        return out

    @staticmethod
    def backward(ctx, grad_out):
        kept, signal = ctx.saved_tensors
        B, T, k, h, halves = ctx.dims
        lib = _lib.load()
        g = grad_out.contiguous()
        grad = torch.empty(k, 3 * h + 1, dtype=kept.dtype, device=kept.device)
        at = kept.data_ptr()
        nets = _pointers([at + 4 * (c * (3 * h + 1) + part * h) for c in range(k) for part in range(4)])
        x = at + 4 * k * (3 * h + 1) if halves else signal.data_ptr()
        with _lib.on_device(kept.device):
            nbytes = lib.ringattr_gain_workspace_bytes(k, h, T, B)
            if nbytes == 0:
                _lib.check(1)
            ws = torch.empty(nbytes, dtype=torch.uint8, device=kept.device)
            _lib.check(lib.ringattr_gain_nets_bwd(x, int(halves), nets, g.data_ptr(), grad.data_ptr(), k, h, T, B, ws.data_ptr(), nbytes,
                                                  _lib.stream_handle(kept.device)))
        parts = list(grad.view(-1).split((h, h, h, 1) * k))
        for c in range(0, 4 * k, 4):
            parts[c], parts[c + 2] = parts[c].view(h, 1), parts[c + 2].view(1, h)
        return (None, None, *parts)


def _pointers(addresses):
    return (ctypes.c_void_p * len(addresses))(*addresses)


def _net_parameters(nets, signal):
    """The parameter tensors as RingGainNetsFunc takes them, or None if these networks or this signal are not its case."""
    if not 1 <= len(nets) <= 16 or signal.dtype != torch.float32 or signal.requires_grad or signal.numel() == 0:
        return None
    h, device = nets[0][0].weight.shape[0], signal.device
    params = []
    for net in nets:
        lin1, lin2 = net[0], net[2]
        for t, shape in ((lin1.weight, (h, 1)), (lin1.bias, (h,)), (lin2.weight, (1, h)), (lin2.bias, (1,))):
            if t is None or t.shape != shape or t.dtype != torch.float32 or t.device != device or not t.is_contiguous():
                return None
            params.append(t)
    return params if 1 <= h <= 32 else None


def ring_gain_nets(base_signal, nets):
    """[B,T,k] base signal through its channels' gain networks (nn.Sequential modules) -> [B,T,k] action signal."""
    params = _net_parameters(nets, base_signal) if base_signal.dim() == 3 and base_signal.shape[2] == len(nets) else None
    if params is None:
        return ring_gain_func(base_signal, pack_gain_nets(nets))
    return RingGainNetsFunc.apply(base_signal.contiguous(), False, *params)


def ring_gain_halves(av_signal, nets):
    """[B,T] angular velocity -> [B,T,2] action signal: relu(-av) and relu(av) through the two networks."""
    params = _net_parameters(nets, av_signal) if av_signal.dim() == 2 and len(nets) == 2 else None
    if params is None:
        base = torch.cat([torch.relu(-av_signal).unsqueeze(2), torch.relu(av_signal).unsqueeze(2)], dim=2)
        return ring_gain_func(base, pack_gain_nets(nets))
    return RingGainNetsFunc.apply(av_signal.contiguous(), True, *params)
