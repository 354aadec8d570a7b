"""GPU tests of the teams of one (17 <= N <= 128, up to six channels: a workgroup per batch tile, weights in registers):
parity with the fp64 oracle at the edges of tiles, chunks and matrix groups, the rebuilt record's bits, rows across batches,
and the fused loss head."""
import numpy as np
import pytest
import torch

from oracle import ring_oracle as O
from tests.ring_cases import make_problem

pytestmark = pytest.mark.gpu

ACTS = {"relu": 0, "gelu": 1, "tanh": 2, "silu": 3}
TRAJ_TOL = 1e-2      # bf16 operands against fp64, as in the parity tests of the other families
GRAD_COS, GRAD_TOL = 0.999, 2e-2

# B, T, k, N, act: two and four chunks, whole and cut; widths 0 to 3 modulo 4; single steps, odd and even lengths; one to six
# channels (both register groups); ragged tiles, one row, more tiles than compute units; 4 rows per workgroup up to 1024, 8 up
# to 2048, then 16, each with both register groups and with odd widths
CASES = [(1, 1, 1, 17, "tanh"), (16, 2, 2, 32, "gelu"), (33, 3, 2, 64, "silu"), (20, 7, 3, 65, "gelu"), (15, 4, 4, 99, "tanh"),
         (64, 9, 2, 120, "tanh"), (50, 6, 6, 126, "gelu"), (40, 5, 5, 127, "silu"), (17, 8, 2, 128, "gelu"), (4200, 3, 2, 101, "gelu"),
         (1500, 5, 2, 101, "gelu"), (1100, 4, 5, 120, "silu"), (1500, 5, 5, 101, "tanh"), (2047, 4, 2, 120, "tanh"), (1030, 3, 3, 50, "gelu"),
         (2101, 5, 5, 127, "silu")]


def _t(x, dev):
    return torch.tensor(x, device=dev)


def _run(p, act, J0, J1, dev, saved=True, ga=True, G=None):
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    A, Wa, Wo, r0 = (_t(p[x], dev) for x in ("A", "Wa", "Wo", "r0"))
    G = _t(p["G"], dev) if G is None else G
    B, T, k = p["A"].shape
    N = p["Wo"].shape[0]
    hist = torch.full((T, B, N), float("nan"), device=dev)
    sv = torch.empty(rnn_cuda.saved_nbytes(N, k, T, B), dtype=torch.uint8, device=dev).fill_(0xFF) if saved else None
    common = dict(A=A, Wa=Wa, J0=J0, J1=J1, Wo=Wo, r_init=r0, bump_history=hist, alpha=0.15, activation_type=ACTS[act], saved=sv)
    rnn_cuda.fwd_cuda.fwd(**common)
    out = {"grad_Wa": torch.full_like(Wa, float("nan")), "grad_Wo": torch.full_like(Wo, float("nan")), "grad_r_init": torch.full_like(r0, float("nan"))}
    if ga:
        out["grad_A"] = torch.full_like(A, float("nan"))
    rnn_cuda.bwd_cuda.bwd(grad_output=G, accumulate=False, **common, **out)
    torch.cuda.synchronize()
    names = _lib.last_kernel_names()
    assert "ring_team_one_fwd" in names["fwd"] and "ring_team_one_bptt" in names["bptt"], names
    return dict(hist=hist, **out)


@pytest.mark.parametrize("B,T,k,N,act", CASES, ids=[f"b{c[0]}_t{c[1]}_k{c[2]}_n{c[3]}" for c in CASES])
def test_teams_of_one_against_the_oracle(B, T, k, N, act, gpu_device):
    print(f"[case] team of one B={B} T={T} k={k} N={N} {act}", flush=True)
    J0, J1 = -1.0 / N, 0.6
    p = make_problem(300 + N + k, B, T, k, N, action="dense")
    got = _run(p, act, J0, J1, gpu_device)
    for other in (_run(p, act, J0, J1, gpu_device), _run(p, act, J0, J1, gpu_device, saved=False), _run(p, act, J0, J1, gpu_device, ga=False)):
        assert not [x for x in other if not torch.equal(got[x], other[x])]       # again; with a rebuilt record; without dL/dA
    ref, _ = O.forward_dense(p["A"], p["Wa"], J0, J1, p["Wo"], p["r0"], 0.15, act)
    assert O.max_rel_err(got["hist"].cpu().numpy(), ref) <= TRAJ_TOL
    g = O.backward_dense(p["G"], p["A"], p["Wa"], J0, J1, p["Wo"], ref, p["r0"], 0.15, act)
    for name in ("grad_Wo", "grad_Wa", "grad_r_init", "grad_A"):
        x = got[name].cpu().numpy()
        assert np.isfinite(x).all(), name
        assert O.cosine(x, g[name]) >= GRAD_COS and O.max_rel_err(x, g[name]) <= GRAD_TOL, name


# 4, 8 and 16 rows per workgroup, whole and cut tiles, both register groups
@pytest.mark.parametrize("B,k,N", [(64, 2, 120), (2048, 2, 128), (1500, 5, 101), (4096, 2, 120), (40, 2, 50)])
def test_teams_of_one_without_a_j0_term_after_a_run_of_nan(B, k, N, gpu_device):
    """J0 = 0: a launch's results do not depend on what an earlier one left in LDS (here operands and row sums of NaN)."""
    print(f"[case] team of one, J0 = 0, B={B} k={k} N={N}", flush=True)
    T = 4
    p = make_problem(500 + N, B, T, k, N, action="dense")
    left = make_problem(501, 4200, 2, k, N, action="dense")
    bad = _run({**left, "r0": np.full_like(left["r0"], np.nan)}, "gelu", -1.0 / N, 0.6, gpu_device)
    assert torch.isnan(bad["hist"]).all() and torch.isnan(bad["grad_r_init"]).all()
    got = _run(p, "gelu", 0.0, 0.6, gpu_device)
    ref, _ = O.forward_dense(p["A"], p["Wa"], 0.0, 0.6, p["Wo"], p["r0"], 0.15, "gelu")
    assert O.max_rel_err(got["hist"].cpu().numpy(), ref) <= TRAJ_TOL
    g = O.backward_dense(p["G"], p["A"], p["Wa"], 0.0, 0.6, p["Wo"], ref, p["r0"], 0.15, "gelu")
    for name in ("grad_Wo", "grad_Wa", "grad_r_init", "grad_A"):
        x = got[name].cpu().numpy()
        assert np.isfinite(x).all(), name
        assert O.cosine(x, g[name]) >= GRAD_COS and O.max_rel_err(x, g[name]) <= GRAD_TOL, name


@pytest.mark.parametrize("N,k", [(100, 2), (127, 5), (50, 3)])
def test_rows_of_teams_of_one_do_not_depend_on_the_batch(N, k, gpu_device):
    B, T = 2300, 6                       # (16 rows per workgroup; the parts have 4 and 8)
    print(f"[case] team of one, rows N={N} k={k}", flush=True)
    p = make_problem(31, B, T, k, N, action="dense")
    whole = _run(p, "gelu", -1.0 / N, 0.6, gpu_device)
    for lo, n in ((0, 1), (5, 16), (37, 100), (16, 512), (1276, 1024), (3, 1025), (250, 2048)):
        part = _run({**p, "A": p["A"][lo:lo + n], "r0": p["r0"][lo:lo + n], "G": p["G"][:, lo:lo + n]}, "gelu", -1.0 / N, 0.6, gpu_device)
        assert torch.equal(part["hist"], whole["hist"][:, lo:lo + n])
        assert torch.equal(part["grad_r_init"], whole["grad_r_init"][lo:lo + n]) and torch.equal(part["grad_A"], whole["grad_A"][lo:lo + n])


@pytest.mark.parametrize("B,T,k,N", [(40, 5, 2, 120), (23, 6, 3, 61)])
def test_fused_loss_head_on_teams_of_one(B, T, k, N, gpu_device):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, ring_rnn_loss_func, ring_loss_pair
    print(f"[case] team of one, loss B={B} T={T} k={k} N={N}", flush=True)
    p = make_problem(77, B, T, k, N, action="dense")
    r0 = _t(p["r0"], gpu_device)
    angle = torch.rand(B, T, device=gpu_device) * 6.28
    grads = []
    for fused in (True, False):
        A, Wa, Wo = (_t(p[x], gpu_device).requires_grad_(True) for x in ("A", "Wa", "Wo"))
        args = (A, Wa, -1.0 / N, 0.6, Wo, r0, 0.15, "gelu")
        total = ring_rnn_loss_func(*args, angle, 0.2)[0] if fused else ring_loss_pair(ring_rnn_cuda_func(*args), angle, 0.2)[0]
        total.backward()
        grads.append((total.detach().cpu().numpy(), A.grad.cpu().numpy(), Wa.grad.cpu().numpy(), Wo.grad.cpu().numpy()))
    assert abs(grads[0][0] - grads[1][0]) <= 1e-5 * abs(grads[1][0])
    # fp32 differences in the loss gradient can flip the bf16 rounding of g: one part in 2^8 of single contributions
    assert all(O.max_rel_err(x, y) <= 4e-3 for x, y in zip(grads[0][1:], grads[1][1:]))
