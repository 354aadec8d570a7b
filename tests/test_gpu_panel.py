"""Panel kernels (wide rings, forward without a saved record): bit for bit the step-per-launch block kernels, whatever
the panel's shape, and the fp64 oracle."""
import numpy as np
import pytest
import torch

from oracle import ring_oracle as O
from ring_cases import make_problem

pytestmark = pytest.mark.gpu


def _forward(p, act, J0, J1, dev):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func
    t = lambda x: torch.as_tensor(x, dtype=torch.float32, device=dev)
    with torch.no_grad():
        return ring_rnn_cuda_func(t(p["A"]), t(p["Wa"]), J0, J1, t(p["Wo"]), t(p["r0"]), 0.15, act)


# rows: one, a full tile and one more, more tiles than a panel holds; neurons: past the team kernels, not a multiple of
# four, the widest; channels: one, two, a fourth column tile's worth, many, more than one pass holds; a silent channel
@pytest.mark.parametrize("B,T,k,N,act,shape", [
    (1, 3, 2, 1025, "relu", None), (17, 3, 1, 1030, "gelu", None), (150, 2, 3, 1536, "tanh", None),
    (40, 2, 16, 2048, "silu", None), (130, 2, 4, 1600, "gelu", "84"), (33, 2, 24, 600, "tanh", None),
    (20, 2, 21, 700, "relu", "22"), (70, 2, 6, 1100, "silu", "42"),
    # what travels between the steps comes round again: more steps than buffers, the last four neurons not whole
    (33, 7, 2, 1027, "gelu", "11"), (20, 8, 2, 1025, "tanh", "24"), (150, 7, 3, 1030, "silu", "81"), (1, 9, 16, 2047, "gelu", None),
    # the most workgroups that do not queue (256), and more
    (32, 5, 2, 2047, "gelu", "11"), (33, 5, 2, 2047, "gelu", "11"), (1000, 4, 16, 1100, "tanh", None),
    # a single step, and two
    (20, 1, 2, 2047, "gelu", None), (130, 1, 7, 768, "silu", None), (130, 2, 7, 768, "silu", None),
])
def test_panel_equals_block_kernels_and_oracle(B, T, k, N, act, shape, gpu_device, monkeypatch):
    print(f"[case] panel B={B} T={T} k={k} N={N} {act} shape={shape}", flush=True)
    J0, J1 = -1.0 / N, 0.5
    p = make_problem(7, B, T, k, N, bump="vm", action="dense")
    if k > 2:
        p["A"][:, :, 1] = 0.0
    for name in ("RINGATTR_PANEL", "RINGATTR_PANEL_SHAPE", "RINGATTR_BLOCK", "RINGATTR_WIDE", "RINGATTR_BLOCK_SHAPE"):
        monkeypatch.delenv(name, raising=False)
    if shape:
        monkeypatch.setenv("RINGATTR_PANEL_SHAPE", shape)
    got = _forward(p, act, J0, J1, gpu_device)
    again = _forward(p, act, J0, J1, gpu_device)
    monkeypatch.setenv("RINGATTR_PANEL", "0")
    block = _forward(p, act, J0, J1, gpu_device)
    assert torch.equal(got, again) and torch.equal(got, block)
    ref, _ = O.forward_dense(p["A"], p["Wa"], J0, J1, p["Wo"], p["r0"], 0.15, act)
    assert O.max_rel_err(got.cpu().numpy(), ref) <= 1e-2     # one bf16 rounding per operand, as everywhere
