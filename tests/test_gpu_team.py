"""GPU tests of the team kernels (several workgroups of one XCD keep the weights on chip and exchange the state through
L2): parity with the fp64 oracle over the shapes they are built in, every output of the backward, the rebuilt record,
the fused loss head, run-to-run reproducibility (a read of state that was not complete would differ between runs), two
streams at once, and the exit taken when a wait runs out."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import ring_oracle as O
from tests.ring_cases import make_problem

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ACTS = {"relu": 0, "gelu": 1, "tanh": 2, "silu": 3}
TRAJ_TOL = 1e-2      # bf16 operands against fp64, as in the parity tests of the other families
GRAD_COS, GRAD_TOL = 0.999, 2e-2

# B, T, k, N, act: K chunks 1 to 32 over four and eight compute waves (even and uneven splits), one to four column tiles
# per member, one to several batch tiles per team, ragged rows and widths (N odd, 2 mod 4), one matrix to sixteen channels
# (matrices in LDS), single step, odd and even lengths
CASES = [
    (9, 4, 1, 17, "tanh"), (33, 1, 2, 33, "gelu"), (20, 7, 2, 100, "silu"), (700, 4, 2, 120, "tanh"), (2300, 3, 3, 126, "gelu"),
    (50, 6, 2, 131, "gelu"), (1, 9, 2, 256, "tanh"), (40, 5, 16, 256, "silu"), (300, 4, 9, 250, "tanh"), (600, 3, 3, 230, "gelu"),
    (24, 6, 2, 257, "silu"), (100, 5, 3, 360, "tanh"), (1100, 3, 2, 500, "gelu"), (260, 3, 16, 512, "silu"), (30, 4, 12, 511, "tanh"),
    (48, 5, 2, 513, "gelu"), (150, 3, 2, 768, "tanh"), (290, 3, 2, 1000, "silu"), (17, 4, 3, 1024, "gelu"),
]


def _t(x, dev):
    return torch.tensor(x, device=dev)


def _run(p, act, J0, J1, dev, saved=True, ga=True, keep_record=False):
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    A, Wa, Wo, r0, G = (_t(p[x], dev) for x in ("A", "Wa", "Wo", "r0", "G"))
    B, T, k = p["A"].shape
    N = p["Wo"].shape[0]
    hist = torch.full((T, B, N), float("nan"), device=dev)
    sv = torch.empty(rnn_cuda.saved_nbytes(N, k, T, B), dtype=torch.uint8, device=dev).fill_(0xFF) if saved else None
    rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=J0, J1=J1, Wo=Wo, r_init=r0, bump_history=hist, alpha=0.15,
                          activation_type=ACTS[act], saved=sv)
    gWa, gWo, gr = torch.full_like(Wa, float("nan")), torch.full_like(Wo, float("nan")), torch.full_like(r0, float("nan"))
    gA = torch.full_like(A, float("nan")) if ga else None
    rnn_cuda.bwd_cuda.bwd(grad_output=G, A=A, Wa=Wa, J0=J0, J1=J1, Wo=Wo, bump_history=hist, r_init=r0, grad_Wa=gWa,
                          grad_Wo=gWo, alpha=0.15, activation_type=ACTS[act], saved=sv, grad_r_init=gr, grad_A=gA,
                          accumulate=False)
    torch.cuda.synchronize()
    names = _lib.last_kernel_names()
    assert "ring_team_bptt" in names["bptt"] and ("ring_team_fwd" in names["fwd"] or not saved)
    return dict(hist=hist, grad_Wa=gWa, grad_Wo=gWo, grad_r_init=gr, **({"grad_A": gA} if ga else {}),
                **({"saved": sv} if saved and keep_record else {}))


@pytest.fixture
def teams(monkeypatch):
    for v in ("RINGATTR_STREAMING", "RINGATTR_ROW_TILES", "RINGATTR_BLOCK", "RINGATTR_WIDE", "RINGATTR_SPLIT_FORWARD",
              "RINGATTR_LDS_WEIGHTS", "RINGATTR_BLOCK_SHAPE", "RINGATTR_CLUSTER", "RINGATTR_CLUSTER_BPTT"):
        monkeypatch.delenv(v, raising=False)
    monkeypatch.setenv("RINGATTR_TEAM", "1")


@pytest.mark.parametrize("B,T,k,N,act", CASES, ids=[f"b{c[0]}_t{c[1]}_k{c[2]}_n{c[3]}" for c in CASES])
def test_team_kernels_against_the_oracle(B, T, k, N, act, gpu_device, teams):
    print(f"[case] team B={B} T={T} k={k} N={N} {act}", flush=True)
    J0, J1 = -1.0 / N, 0.6
    p = make_problem(900 + N + k, B, T, k, N, action="dense")
    if k > 3:
        p["A"][:, :, k // 2] = 0.0         # one silent channel among the driven ones
    got = _run(p, act, J0, J1, gpu_device)
    again = _run(p, act, J0, J1, gpu_device)
    assert all(torch.equal(got[x], again[x]) for x in got)
    rebuilt = _run(p, act, J0, J1, gpu_device, saved=False)
    plain = _run(p, act, J0, J1, gpu_device, ga=False)
    assert all(torch.equal(got[x], rebuilt[x]) for x in got if x != "hist")     # the same recurrence, run again
    assert all(torch.equal(got[x], plain[x]) for x in plain)
    ref, _ = O.forward_dense(p["A"], p["Wa"], J0, J1, p["Wo"], p["r0"], 0.15, act)
    assert O.max_rel_err(got["hist"].cpu().numpy(), ref) <= TRAJ_TOL
    g = O.backward_dense(p["G"], p["A"], p["Wa"], J0, J1, p["Wo"], ref, p["r0"], 0.15, act)
    for name in ("grad_Wo", "grad_Wa", "grad_r_init", "grad_A"):
        x = got[name].cpu().numpy()
        assert np.isfinite(x).all(), name
        assert O.cosine(x, g[name]) >= GRAD_COS and O.max_rel_err(x, g[name]) <= GRAD_TOL, name


# two and four items per workgroup of the rebuild, odd and even lengths, ragged rows and widths, channels that are silent
@pytest.mark.parametrize("B,T,k,N,act", [(9, 1, 1, 17, "gelu"), (700, 48, 2, 120, "tanh"), (530, 65, 3, 131, "silu"),
                                         (100, 9, 3, 360, "gelu"), (1030, 32, 16, 250, "tanh"), (40, 6, 2, 1000, "silu")])
def test_backward_without_a_record_differentiates_the_history_it_is_given(B, T, k, N, act, gpu_device, teams):
    """The reference's boundary hands the backward a history and no record; the record follows from that history whoever
    made it, so every gradient is the given trajectory's."""
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    print(f"[case] team rebuild B={B} T={T} k={k} N={N} {act}", flush=True)
    J0, J1 = -1.0 / N, 0.6
    p = make_problem(500 + N + k, B, T, k, N, action="dense")
    if k > 3:
        p["A"][:, :, 2:] = 0.0
    hist, _ = O.forward_dense(p["A"], p["Wa"], J0, J1, p["Wo"], p["r0"], 0.15, act)
    rng = np.random.default_rng(B + T)
    hist = (hist * (1.0 + 0.3 * rng.standard_normal(hist.shape)) + 0.02 * rng.standard_normal(hist.shape)).astype(np.float32)
    A, Wa, Wo, r0, G, H = (_t(x, gpu_device) for x in (p["A"], p["Wa"], p["Wo"], p["r0"], p["G"], hist))
    got = {n: torch.full_like(x, float("nan")) for n, x in (("grad_Wa", Wa), ("grad_Wo", Wo), ("grad_r_init", r0), ("grad_A", A))}
    rnn_cuda.bwd_cuda.bwd(grad_output=G, A=A, Wa=Wa, J0=J0, J1=J1, Wo=Wo, bump_history=H, r_init=r0, alpha=0.15,
                          activation_type=ACTS[act], accumulate=False, **got)
    torch.cuda.synchronize()
    want = O.backward_dense(p["G"], p["A"], p["Wa"], J0, J1, p["Wo"], hist.astype(np.float64), p["r0"], 0.15, act)
    for name, x in got.items():
        x = x.cpu().numpy()
        assert np.isfinite(x).all(), name
        assert O.cosine(x, want[name]) >= GRAD_COS and O.max_rel_err(x, want[name]) <= GRAD_TOL, name
    names = _lib.last_kernel_names()
    assert "ring_team_rebuild" in names["rebuild_saved"] and "ring_team_bptt" in names["bptt"], names


@pytest.mark.parametrize("N,B,T,act", [(256, 1, 100, "gelu"), (256, 512, 21, "tanh"), (256, 100, 2, "relu"), (129, 16, 40, "silu"),
                                       (131, 9, 1, "gelu"), (200, 257, 33, "gelu"), (250, 300, 12, "tanh"), (222, 64, 17, "relu")])
def test_small_batches_without_a_record_have_the_weight_resident_forwards_bits(N, B, T, act, gpu_device, teams, monkeypatch):
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    print(f"[case] team rows N={N} B={B} T={T} {act}", flush=True)
    p = make_problem(85, B, T, 2, N, action="dense")
    A, Wa, Wo, r0 = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0"))

    def fwd(kernel, **env):
        monkeypatch.delenv("RINGATTR_TEAM", raising=False)
        for name, value in env.items():
            monkeypatch.setenv(name, value)
        out = torch.full((T, B, N), float("nan"), device=gpu_device)
        rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-0.05, J1=0.7, Wo=Wo, r_init=r0, bump_history=out, alpha=0.15, activation_type=ACTS[act])
        torch.cuda.synchronize()
        for name in env:
            monkeypatch.delenv(name)
        assert kernel in _lib.last_kernel_names()["fwd"]
        return out

    want = fwd("ring_fwd_res256", RINGATTR_TEAM="0")
    assert torch.isfinite(want).all()
    for wait_us in (None, "-1", "0"):
        for _ in range(3):
            got = fwd("ring_team_rows", **({} if wait_us is None else {"RINGATTR_TEAM_GATHER_US": wait_us}))
            assert torch.equal(got, want), wait_us


# rings with teams for more than 512 rows as long as no record is wanted: the most of each number of members, and one more
@pytest.mark.parametrize("N,B,kernel", [(129, 513, "ring_team_rows"), (160, 768, "ring_team_rows"), (160, 769, "ring_fwd_res256"),
                                        (192, 640, "ring_team_rows"), (192, 641, "ring_fwd_res256"), (193, 513, "ring_fwd_res256")])
def test_forwards_without_a_record_take_teams_as_far_as_they_go(N, B, kernel, gpu_device, monkeypatch):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, _lib
    monkeypatch.delenv("RINGATTR_TEAM", raising=False)
    print(f"[case] team rows as far as they go N={N} B={B}", flush=True)
    p = make_problem(86, B, 3, 2, N, action="dense")
    args = [_t(p["A"], gpu_device), _t(p["Wa"], gpu_device), -0.05, 0.7, _t(p["Wo"], gpu_device), _t(p["r0"], gpu_device), 0.15, "gelu"]
    with torch.no_grad():
        got = ring_rnn_cuda_func(*args)
        assert kernel in _lib.last_kernel_names()["fwd"]
        monkeypatch.setenv("RINGATTR_TEAM", "0")
        assert torch.equal(got, ring_rnn_cuda_func(*args))


# the kernels of 128 < N <= 256 with two channels, whole and ragged widths; teams with members of different width per batch
@pytest.mark.parametrize("N,k,B,kernel", [(256, 2, 4096, "res256"), (200, 2, 1500, "res256"), (120, 2, 4096, "team"),
                                          (360, 2, 2048, "team"), (333, 3, 1000, "team"), (700, 2, 1024, "team")])
def test_rows_do_not_depend_on_the_batch_they_are_in(N, k, B, kernel, gpu_device, teams, monkeypatch):
    """A slice of a batch run alone reproduces its rows of the full batch bit for bit, whatever its size.  (At N = 256 the
    weight-resident BPTT of ragged batches is another variant than that of whole tiles: dL/dr_init is compared there for
    whole tiles.)"""
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, _lib
    monkeypatch.delenv("RINGATTR_TEAM")
    T = 9
    print(f"[case] rows across batches N={N} k={k} B={B}", flush=True)
    p = make_problem(84, B, T, k, N, action="dense")
    G = torch.randn(T, B, N, device=gpu_device, generator=torch.Generator(device=gpu_device).manual_seed(5))
    Wa, Wo = _t(p["Wa"], gpu_device).requires_grad_(True), _t(p["Wo"], gpu_device).requires_grad_(True)

    def run(rows):
        A, r0 = _t(p["A"][rows], gpu_device), _t(p["r0"][rows], gpu_device).requires_grad_(True)
        hist = ring_rnn_cuda_func(A, Wa, -1.0 / N, 0.6, Wo, r0, 0.15, "gelu")
        hist.backward(G[:, rows].contiguous())
        names = _lib.last_kernel_names()
        assert kernel in names["fwd"] and kernel in names["bptt"], names
        with torch.no_grad():
            assert torch.equal(ring_rnn_cuda_func(A, Wa, -1.0 / N, 0.6, Wo, r0, 0.15, "gelu"), hist)     # and without a record
        return hist.detach(), r0.grad

    full = run(slice(0, B))
    for lo, n in ((5, 1), (16, 16), (3, 100), (128, 128), (0, B // 2), (0, 1000 if B > 1000 else 500)):
        part = run(slice(lo, lo + n))
        assert torch.equal(part[0], full[0][:, lo:lo + n]), (lo, n)
        if N != 256 or n % 16 == 0:
            assert torch.equal(part[1], full[1][lo:lo + n]), (lo, n)


@pytest.mark.parametrize("B,T,k,N", [(40, 7, 2, 120), (20, 6, 16, 100), (100, 5, 3, 360), (300, 4, 2, 700)])
def test_backward_stays_inside_the_workspace_it_asks_for(B, T, k, N, gpu_device, teams):
    """The areas that take turns in the workspace, against the workspace's end and against each other: same bits as with
    room to spare, nothing written behind the end."""
    from rnn_train_ring_attractor_amd import _lib, rnn_cuda
    print(f"[case] team workspace B={B} T={T} k={k} N={N}", flush=True)
    lib = _lib.load()
    p = make_problem(83, B, T, k, N, action="dense")
    A, Wa, Wo, r0, G = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0", "G"))
    hist = torch.empty(T, B, N, device=gpu_device)
    record = torch.empty(rnn_cuda.saved_nbytes(N, k, T, B), dtype=torch.uint8, device=gpu_device)
    rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-0.01, J1=0.6, Wo=Wo, r_init=r0, bump_history=hist, alpha=0.15, activation_type=1, saved=record)
    for saved in (record, None):
        for ga in (False, True):
            need = lib.ringattr_bwd_workspace_bytes_for(N, k, T, B, int(saved is not None), int(ga))

            def bwd(space, nbytes):
                out = [torch.full_like(x, float("nan")) for x in (Wa, Wo, r0)] + ([torch.full_like(A, float("nan"))] if ga else [])
                ptr = lambda x: None if x is None else x.data_ptr()
                rc = lib.ringattr_bwd(ptr(G), ptr(A), ptr(Wa), -0.01, 0.6, ptr(Wo), ptr(hist), ptr(r0), ptr(out[0]), ptr(out[1]), 0.15,
                                      N, k, T, B, 1, 0, ptr(saved), ptr(out[3]) if ga else None, ptr(out[2]), ptr(space), nbytes,
                                      torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                return rc, out

            roomy = torch.zeros(2 * need + (1 << 20), dtype=torch.uint8, device=gpu_device)
            tight = torch.full((need + 4096,), 0xAB, dtype=torch.uint8, device=gpu_device)
            (rc0, want), (rc1, got) = bwd(roomy, roomy.numel()), bwd(tight, need)
            assert rc0 == 0 and rc1 == 0 and "ring_team_bptt" in _lib.last_kernel_names()["bptt"]
            assert all(torch.equal(x, y) for x, y in zip(got, want)) and bool((tight[need:] == 0xAB).all())


# Sequences that go through the exchange slots many times: one tile per team (8 slots), teams of one and two tiles and of
# two (6 slots), of three and four (4 slots, the fullest and the others), sixteen; the sizes of ordinary calls among them
@pytest.mark.parametrize("B,T,k,N", [(64, 120, 2, 120), (100, 75, 3, 360), (150, 50, 2, 600), (1000, 45, 2, 360), (256, 20, 16, 512),
                                     (400, 44, 2, 1000), (2048, 120, 2, 1024)])
def test_slots_are_reused_many_times(B, T, k, N, gpu_device, teams, monkeypatch):
    """A slot of the exchange area is emptied and published again every 8, 6 or 4 steps.  Single workgroups, which exchange
    nothing, give the same bits; row-wise outputs are held to the fp64 oracle on rows of the first tile, the last one and
    one of a team with fewest tiles."""
    print(f"[case] team slots B={B} T={T} k={k} N={N}", flush=True)
    J0, J1 = -1.0 / N, 0.6
    p = make_problem(86, B, T, k, N, action="dense")
    # (dL/dA of the largest shape would need a share per member of all its steps)
    got = _run(p, "tanh", J0, J1, gpu_device, ga=B < 2048)
    monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")
    alone = _run(p, "tanh", J0, J1, gpu_device, ga=B < 2048)
    monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
    assert all(torch.equal(got[x], alone[x]) for x in got), [x for x in got if not torch.equal(got[x], alone[x])]
    del alone
    again = _run(p, "tanh", J0, J1, gpu_device, ga=B < 2048)
    assert all(torch.equal(got[x], again[x]) for x in got)
    del again
    rows = np.array(sorted({0, 7, B // 2, B - 1} | {r for r in (16 * 7 + 3, 16 * 15 + 9, 16 * 39 + 1) if r < B}))
    ref, _ = O.forward_dense(p["A"][rows], p["Wa"], J0, J1, p["Wo"], p["r0"][rows], 0.15, "tanh")
    assert O.max_rel_err(got["hist"][:, torch.as_tensor(rows, device=gpu_device)].cpu().numpy(), ref) <= TRAJ_TOL
    g = O.backward_dense(p["G"][:, rows], p["A"][rows], p["Wa"], J0, J1, p["Wo"], ref, p["r0"][rows], 0.15, "tanh")
    for name in [x for x in ("grad_r_init", "grad_A") if x in got]:
        x = got[name][torch.as_tensor(rows, device=gpu_device)].cpu().numpy()
        assert O.cosine(x, g[name]) >= GRAD_COS and O.max_rel_err(x, g[name]) <= GRAD_TOL, name


@pytest.mark.parametrize("B,T,k,N", [(40, 5, 2, 120), (70, 6, 3, 361)])
def test_fused_loss_head_on_teams(B, T, k, N, gpu_device, teams):
    """The objective's gradient formed inside the team BPTT against the loss head's own backward through the plain one."""
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, ring_rnn_loss_func, ring_loss_pair
    print(f"[case] team loss B={B} T={T} k={k} N={N}", flush=True)
    p = make_problem(77, B, T, k, N, action="dense")
    A, r0 = _t(p["A"], gpu_device), _t(p["r0"], gpu_device)
    angle = torch.rand(B, T, device=gpu_device) * 6.28
    grads = []
    for fused in (True, False):
        Wa, Wo = _t(p["Wa"], gpu_device).requires_grad_(True), _t(p["Wo"], gpu_device).requires_grad_(True)
        if fused:
            total = ring_rnn_loss_func(A, Wa, -1.0 / N, 0.6, Wo, r0, 0.15, "gelu", angle, 0.2)[0]
        else:
            total = ring_loss_pair(ring_rnn_cuda_func(A, Wa, -1.0 / N, 0.6, Wo, r0, 0.15, "gelu"), angle, 0.2)[0]
        total.backward()
        grads.append((float(total), Wa.grad.cpu().numpy(), Wo.grad.cpu().numpy()))
    assert abs(grads[0][0] - grads[1][0]) <= 1e-5 * abs(grads[1][0])
    # fp32 differences in the loss gradient can flip the bf16 rounding of g: one part in 2^8 of single contributions
    assert O.max_rel_err(grads[0][1], grads[1][1]) <= 4e-3 and O.max_rel_err(grads[0][2], grads[1][2]) <= 4e-3


def test_teams_on_two_streams(gpu_device, teams):
    """Two launches that each want compute units of the whole device, issued on two streams: the second waits for the
    first instead of sharing the device with it half and half, and both give the sequential result."""
    B, T, k, N = 600, 24, 2, 512
    print(f"[case] teams on two streams B={B} T={T} N={N}", flush=True)
    from rnn_train_ring_attractor_amd import rnn_cuda
    p = make_problem(78, B, T, k, N, action="dense")
    A, Wa, Wo, r0 = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0"))

    def fwd(out):
        rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-1.0 / N, J1=0.6, Wo=Wo, r_init=r0, bump_history=out, alpha=0.15, activation_type=2)

    ref = torch.empty(T, B, N, device=gpu_device)
    fwd(ref)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=gpu_device) for _ in range(2)]
    outs = [torch.full((T, B, N), float("nan"), device=gpu_device) for _ in range(6)]
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        with torch.cuda.stream(streams[i % 2]):
            fwd(o)
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
    fwd(ref)                       # (a wait that had run out would be reported by this call)


@pytest.mark.parametrize("B,T,k,N,act", CASES + [(40, 5, 2, 120, "relu")], ids=[f"b{c[0]}_t{c[1]}_k{c[2]}_n{c[3]}" for c in CASES] + ["relu"])
def test_teams_that_do_not_gather_are_done_by_single_workgroups_with_the_same_bits(B, T, k, N, act, gpu_device, teams, monkeypatch):
    """A team whose members do not become resident together (another team launch may hold the compute units they lack)
    gives up before the time loop, and a launch behind does its tiles.  Here the host lets every team give up at once, and
    then after no wait at all, when some teams are complete and others are not."""
    print(f"[case] ungathered teams B={B} T={T} k={k} N={N} {act}", flush=True)
    p = make_problem(900 + N + k, B, T, k, N, action="dense")
    if k > 3:
        p["A"][:, :, k // 2] = 0.0
    for ga in (True, False):
        want = _run(p, act, -1.0 / N, 0.6, gpu_device, ga=ga, keep_record=True)
        for wait_us in ("-1", "0", "2"):
            monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", wait_us)
            got = _run(p, act, -1.0 / N, 0.6, gpu_device, ga=ga, keep_record=True)
            monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
            assert all(torch.equal(got[x], want[x]) for x in want), [x for x in want if not torch.equal(got[x], want[x])]


def test_objective_of_teams_that_do_not_gather(gpu_device, teams, monkeypatch):
    from rnn_train_ring_attractor_amd import ring_rnn_loss_func
    B, T, k, N = 70, 6, 3, 361
    print(f"[case] ungathered teams, objective B={B} T={T} k={k} N={N}", flush=True)
    p = make_problem(77, B, T, k, N, action="dense")
    r0 = _t(p["r0"], gpu_device)
    angle = torch.rand(B, T, device=gpu_device) * 6.28
    for want_a in (False, True):
        runs = []
        for wait_us in ("50000", "-1"):
            monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", wait_us)
            leaves = [_t(p[x], gpu_device).requires_grad_(x != "A" or want_a) for x in ("A", "Wa", "Wo")]
            total = ring_rnn_loss_func(leaves[0], leaves[1], -1.0 / N, 0.6, leaves[2], r0, 0.15, "gelu", angle, 0.2)[0]
            total.backward()
            runs.append([total.detach()] + [x.grad for x in leaves if x.grad is not None])
        assert len(runs[0]) == (4 if want_a else 3) and all(torch.equal(x, y) for x, y in zip(*runs))


def test_cluster_and_team_launches_on_two_streams(gpu_device, teams, monkeypatch):
    """Teams of 32 on one stream and the N = 512 clusters on another, launched in turn: between them they could fill an XCD
    with workgroups that wait for others, so they run one after the other."""
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    monkeypatch.delenv("RINGATTR_TEAM")
    jobs = []
    for B, T, N, kernel in ((8192, 16, 512, "ring_fwd_cluster8"), (128, 40, 1000, "ring_team_fwd")):
        p = make_problem(82, B, T, 2, N, action="dense")
        A, Wa, Wo, r0 = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0"))

        def fwd(out, A=A, Wa=Wa, Wo=Wo, r0=r0, N=N):
            rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-1.0 / N, J1=0.6, Wo=Wo, r_init=r0, bump_history=out, alpha=0.15, activation_type=2)

        ref = torch.empty(T, B, N, device=gpu_device)
        fwd(ref)
        assert kernel in _lib.last_kernel_names()["fwd"]
        jobs.append((fwd, ref, torch.cuda.Stream(device=gpu_device), [torch.full_like(ref, float("nan")) for _ in range(3)]))
    print("[case] clusters and teams on two streams", flush=True)
    torch.cuda.synchronize()
    for i in range(3):
        for fwd, _, st, outs in jobs:
            with torch.cuda.stream(st):
                fwd(outs[i])
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for _, ref, _, outs in jobs for o in outs)
    jobs[0][0](jobs[0][1])         # (a wait that had run out would be reported by this call)


def test_graphs_replayed_on_two_streams(gpu_device, teams):
    """Nothing on the host orders the team launches of two replayed graphs.  Each of these wants every compute unit for its
    teams of 32; whichever teams starve give up and are done by single workgroups."""
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    B, T, k, N = 128, 12, 2, 1000
    print(f"[case] two graphs of team forwards on two streams B={B} T={T} N={N}", flush=True)
    p = make_problem(81, B, T, k, N, action="dense")
    A, Wa, Wo, r0 = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0"))

    def fwd(out):
        rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-1.0 / N, J1=0.6, Wo=Wo, r_init=r0, bump_history=out, alpha=0.15, activation_type=2)

    ref = torch.empty(T, B, N, device=gpu_device)
    fwd(ref)
    assert "ring_team_fwd" in _lib.last_kernel_names()["fwd"]
    outs = [torch.empty_like(ref) for _ in range(2)]
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for g, o in zip(graphs, outs):
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            fwd(o)
    streams = [torch.cuda.Stream(device=gpu_device) for _ in range(2)]
    for _ in range(4):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        for st, g in zip(streams, graphs):
            with torch.cuda.stream(st):
                g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, ref) for o in outs)
    fwd(ref)                       # (a wait that had run out would be reported by this call)


_GIVE_UP_SCRIPT = r"""
import os, sys
sys.path.insert(0, {root!r})
os.environ["RINGATTR_TEAM"] = "1"
os.environ["RINGATTR_CLUSTER_SPIN"] = "-1"      # every wave gives up its waits at once
import torch
from tests.ring_cases import make_problem
from rnn_train_ring_attractor_amd import rnn_cuda, _lib
dev = torch.device("cuda:0")
p = make_problem(315, 64, 6, 2, 360, action="dense")
A, Wa, Wo, r0 = (torch.tensor(p[k], device=dev) for k in ("A", "Wa", "Wo", "r0"))
def fwd():
    hist = torch.full((6, 64, 360), float("nan"), device=dev)
    rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-0.01, J1=0.5, Wo=Wo, r_init=r0, bump_history=hist, alpha=0.15, activation_type=2)
    torch.cuda.synchronize()
    return hist
print("[case] team forward whose waves give up", flush=True)
fwd()                                             # the launch goes through its steps without waiting and ends
assert "team" in _lib.last_kernel_names()["fwd"]
try:
    fwd()
    sys.exit(1)
except Exception as e:                            # reported once, by the next call
    assert "gave up waiting" in str(e), str(e)
h = fwd()                                         # from here on the other kernels do the work
assert "team" not in _lib.last_kernel_names()["fwd"] and torch.isfinite(h).all()
print("give-up path ok")
"""


def test_a_wait_that_runs_out_is_reported_once_and_the_other_kernels_take_over(gpu_device):
    proc = subprocess.run([sys.executable, "-c", _GIVE_UP_SCRIPT.format(root=ROOT)], capture_output=True, text=True, timeout=300,
                          cwd=ROOT)
    print(proc.stdout[-1500:], proc.stderr[-1500:], flush=True)
    assert proc.returncode == 0 and "give-up path ok" in proc.stdout


# one row to all 32 teams, ragged tiles and widths (padding within a chunk, whole chunks of it), single steps, odd and even lengths
@pytest.mark.parametrize("N,B,T,act", [(256, 1, 7, "gelu"), (256, 128, 100, "gelu"), (256, 512, 12, "tanh"), (256, 40, 2, "silu"), (129, 16, 1, "silu"),
                                       (131, 9, 3, "gelu"), (200, 257, 33, "gelu"), (250, 300, 6, "tanh"), (222, 64, 17, "relu")])
def test_small_batches_train_with_the_weight_resident_kernels_bits(N, B, T, act, gpu_device, teams, monkeypatch):
    """Forward with a record and BPTT over teams against the weight-resident kernels, every output; either family's record
    through the other one's BPTT; and the single workgroups behind teams that do not gather."""
    from rnn_train_ring_attractor_amd import rnn_cuda, _lib
    monkeypatch.delenv("RINGATTR_TEAM", raising=False)
    print(f"[case] team rows, training N={N} B={B} T={T} {act}", flush=True)
    p = make_problem(87, B, T, 2, N, action="dense")
    A, Wa, Wo, r0, G = (_t(p[x], gpu_device) for x in ("A", "Wa", "Wo", "r0", "G"))
    common = dict(A=A, Wa=Wa, J0=-0.05, J1=0.7, Wo=Wo, r_init=r0, alpha=0.15, activation_type=ACTS[act])

    def fwd(kernel, **env):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        hist = torch.full((T, B, N), float("nan"), device=gpu_device)
        saved = torch.empty(rnn_cuda.saved_nbytes(N, 2, T, B), dtype=torch.uint8, device=gpu_device).fill_(0xFF)
        rnn_cuda.fwd_cuda.fwd(bump_history=hist, saved=saved, **common)
        torch.cuda.synchronize()
        for k in env:
            monkeypatch.delenv(k)
        assert kernel in _lib.last_kernel_names()["fwd"]
        return hist, saved

    def bwd(kernel, hist, saved, ga, **env):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        out = {n: torch.full_like(x, float("nan")) for n, x in (("grad_Wa", Wa), ("grad_Wo", Wo), ("grad_r_init", r0))}
        if ga:
            out["grad_A"] = torch.full_like(A, float("nan"))
        rnn_cuda.bwd_cuda.bwd(grad_output=G, bump_history=hist, saved=saved, accumulate=False, **common, **out)
        torch.cuda.synchronize()
        for k in env:
            monkeypatch.delenv(k)
        assert kernel in _lib.last_kernel_names()["bptt"]
        return out

    resident, team = dict(RINGATTR_TEAM="0"), {}
    hist, record = fwd("ring_fwd_res256", **resident)
    assert torch.isfinite(hist).all()
    for ga in (True, False):
        want = bwd("ring_bptt_res256", hist, record, ga, **resident)
        for wait_us in (None, "-1", "0"):
            env = {} if wait_us is None else {"RINGATTR_TEAM_GATHER_US": wait_us}
            h, s = fwd("ring_team_res256_fwd", **env)
            assert torch.equal(h, hist), wait_us
            for got in (bwd("ring_team_res256_bptt", h, s, ga, **env), bwd("ring_bptt_res256", h, s, ga, **resident),
                        bwd("ring_team_res256_bptt", hist, record, ga, **env)):
                bad = {x: float((got[x] - want[x]).abs().max() / want[x].abs().max()) for x in want if not torch.equal(got[x], want[x])}
                assert not bad, (wait_us, ga, bad)


# whole and ragged tiles, single steps: the row sums' order and the late columns' record
@pytest.mark.parametrize("N,B,T,act", [(256, 128, 100, "gelu"), (256, 48, 9, "tanh"), (256, 16, 1, "gelu"), (256, 40, 5, "gelu"), (256, 64, 6, "relu"),
                                       (200, 100, 6, "tanh"), (131, 32, 4, "silu")])
def test_fused_loss_head_on_small_batches_of_the_weight_resident_widths(N, B, T, act, gpu_device, teams, monkeypatch):
    """The loss and every gradient, bit for bit."""
    from rnn_train_ring_attractor_amd import ring_rnn_loss_func, _lib
    print(f"[case] team rows, loss N={N} B={B} T={T} {act}", flush=True)
    p = make_problem(77, B, T, 2, N, action="dense")
    r0 = _t(p["r0"], gpu_device)
    angle = torch.rand(B, T, device=gpu_device) * 6.28

    def run(**env):
        monkeypatch.delenv("RINGATTR_TEAM", raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        leaves = [_t(p[x], gpu_device).requires_grad_(True) for x in ("A", "Wa", "Wo")]
        out = ring_rnn_loss_func(leaves[0], leaves[1], -1.0 / N, 0.6, leaves[2], r0, 0.15, act, angle, 0.2)
        out[0].backward()
        torch.cuda.synchronize()
        for k in env:
            monkeypatch.delenv(k)
        return [x.detach() for x in out] + [x.grad for x in leaves]

    want = run(RINGATTR_TEAM="0")
    assert "ring_bptt_res256" in _lib.last_kernel_names()["bptt"]
    for env in ({}, {"RINGATTR_TEAM_GATHER_US": "-1"}):
        got = run(**env)
        assert "ring_team_res256_bptt" in _lib.last_kernel_names()["bptt"]
        assert [torch.equal(x, y) for x, y in zip(got, want)] == [True] * len(want), env


@pytest.mark.parametrize("N,B,k", [(112, 40, 16), (144, 33, 12), (300, 200, 16), (385, 20, 7)])
def test_channels_that_are_silent_in_some_items(N, B, k, gpu_device):
    """Matrices in LDS are passed by where their channels are silent in an item's 16 rows: none driven, only the last, only in some
    rows, gates of minus zero; against the oracle (bf16 operands: the bounds of the parity tests)."""
    from oracle import ring_oracle as O
    from tests.ring_cases import make_problem
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func
    T = 6
    print(f"[case] silent channels N={N} B={B} k={k}", flush=True)
    p = make_problem(500 + N, B, T, k, N, action="dense")
    A = p["A"]
    A[:, 0, 2:] = 0.0
    A[:16, 1, :-1] = 0.0
    A[16:, 2, 3:] = -0.0
    A[1:, 3, -1] = 0.0
    A[:, 4, :] = 0.0
    t = lambda x: torch.tensor(x, device=gpu_device)
    Wa, Wo = t(p["Wa"]).requires_grad_(True), t(p["Wo"]).requires_grad_(True)
    hist = ring_rnn_cuda_func(t(A), Wa, -0.05, 0.4, Wo, t(p["r0"]), 0.15, "gelu")
    hist.backward(t(p["G"]))
    torch.cuda.synchronize()
    ref, _ = O.forward_dense(A, p["Wa"], -0.05, 0.4, p["Wo"], p["r0"], 0.15, "gelu")
    g = O.backward_dense(p["G"], A, p["Wa"], -0.05, 0.4, p["Wo"], ref, p["r0"], 0.15, "gelu")
    assert O.max_rel_err(hist.detach().cpu().numpy(), ref) <= 1e-2
    for got, want in ((Wo.grad, g["grad_Wo"]), (Wa.grad, g["grad_Wa"])):
        assert O.cosine(got.cpu().numpy(), want) >= 0.999 and O.max_rel_err(got.cpu().numpy(), want) <= 2e-2


# a case for every kernel that is built for an exact number of matrices in LDS (K chunks 1 to 4 a wave, one to four column tiles a
# member, three or nine matrices in registers)
@pytest.mark.parametrize("B,k,N", [
    (9, 3, 144), (9, 4, 144), (9, 5, 144), (9, 9, 144), (521, 3, 200), (777, 4, 200), (777, 5, 200), (777, 6, 200), (1545, 3, 200), (1545, 4, 200),
    (2313, 5, 144), (9, 3, 260), (9, 4, 260), (9, 5, 260), (9, 9, 260), (393, 3, 260), (393, 4, 260), (265, 5, 290), (265, 6, 260), (9, 3, 520),
    (9, 4, 520), (9, 3, 800)])
def test_few_matrices_in_lds(B, k, N, gpu_device, teams, monkeypatch):
    """Their channels all driven, one of them silent, all of them silent, gates of minus zero: the bits of the single workgroups, and the
    oracle for the first rows."""
    print(f"[case] few matrices in LDS B={B} k={k} N={N}", flush=True)
    T = 5
    p = make_problem(700 + N + k, B, T, k, N, action="dense")
    A = p["A"]
    A[:, 1, 2:] = 0.0
    A[:16, 2, -1] = -0.0
    A[:, 3, -2:-1] = 0.0
    for ga in (True, False):
        want = _run(p, "gelu", -1.0 / N, 0.6, gpu_device, ga=ga)
        monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")
        got = _run(p, "gelu", -1.0 / N, 0.6, gpu_device, ga=ga)
        monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
        assert all(torch.equal(got[x], want[x]) for x in want), [x for x in want if not torch.equal(got[x], want[x])]
    ref, _ = O.forward_dense(A[:9], p["Wa"], -1.0 / N, 0.6, p["Wo"], p["r0"][:9], 0.15, "gelu")
    assert O.max_rel_err(want["hist"][:, :9].cpu().numpy(), ref) <= TRAJ_TOL


# Teams for the weight-resident widths: members of one column tile while every batch tile finds room for a team of them, two past that:
# 256 rows with a record, up to 384 without (five chunks are ten members).
@pytest.mark.parametrize("N,T,act", [(256, 9, "gelu"), (200, 8, "relu"), (131, 5, "silu")])
def test_rows_on_either_side_of_the_line_between_one_and_two_column_tiles(N, T, act, gpu_device, monkeypatch):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, _lib
    p = make_problem(31, 257, T, 2, N)
    t = lambda x: torch.as_tensor(x, dtype=torch.float32, device=gpu_device)
    A, Wa, Wo, r0, G = (t(p[n]) for n in ("A", "Wa", "Wo", "r0", "G"))

    def run(B, **env):
        for name in ("RINGATTR_TEAM", "RINGATTR_TEAM_GATHER_US"):
            monkeypatch.delenv(name, raising=False)
        for name, value in env.items():
            monkeypatch.setenv(name, value)
        a, ra = A[:B].clone().requires_grad_(True), r0[:B].clone()
        with torch.no_grad():
            plain = ring_rnn_cuda_func(a.detach(), Wa, -1.0 / N, 0.5, Wo, ra, 0.15, act)
        wo, wa = Wo.clone().requires_grad_(True), Wa.clone().requires_grad_(True)
        h = ring_rnn_cuda_func(a, wa, -1.0 / N, 0.5, wo, ra, 0.15, act)
        h.backward(G[:, :B].contiguous())
        assert torch.equal(plain, h)
        return h.detach(), a.grad, wo.grad, wa.grad, _lib.last_kernel_names()["bptt"]

    for B in (1, 16, 256, 257):
        teams = run(B)
        assert teams[4].startswith("ring_team_res256_bptt")
        for other in (run(B, RINGATTR_TEAM="0"), run(B, RINGATTR_TEAM_GATHER_US="-1")):      # one workgroup a tile; teams that give up
            for got, want in zip(teams[:4], other[:4]):
                assert torch.equal(got, want), (B, other[4])


# Without a record a team has as many members as the ring has column tiles: ten up to N = 160, three teams an XCD, 384 rows; twelve up to
# N = 192 and more up to 256, two teams an XCD, 256 rows.  With one always sixteen.
@pytest.mark.parametrize("N,rows", [(131, 384), (160, 384), (161, 256), (256, 256)])
def test_members_have_one_column_tile_as_far_as_there_is_room(N, rows, gpu_device, monkeypatch):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, _lib
    p = make_problem(32, 385, 4, 2, N)
    t = lambda x: torch.as_tensor(x, dtype=torch.float32, device=gpu_device)
    A, Wa, Wo, r0 = (t(p[n]) for n in ("A", "Wa", "Wo", "r0"))

    def run(B, record):
        a, r, wo = A[:B].clone(), r0[:B].clone(), Wo.clone().requires_grad_(record)
        return ring_rnn_cuda_func(a, Wa, -1.0 / N, 0.5, wo, r, 0.15, "tanh").detach(), _lib.last_kernel_names()["fwd"]

    for record, kernel, limit in ((False, "ring_team_rows_kernel", rows), (True, "ring_team_res256_fwd_kernel", 256)):
        monkeypatch.delenv("RINGATTR_TEAM", raising=False)
        (one, name_one), (two, name_two) = run(limit, record), run(limit + 1, record)
        assert (name_one, name_two) == (kernel + "<2,1>", kernel + "<2,2>")
        monkeypatch.setenv("RINGATTR_TEAM", "0")
        whole, name = run(limit + 1, record)
        assert not name.startswith("ring_team")
        assert torch.equal(two, whole) and torch.equal(one, whole[:, :limit])


# One column tile a member takes twice the compute units two do.  So only while the launches of other streams that have not finished leave
# room for it (two side by side up to 128 rows), and under capture, where nobody knows what the graph will be replayed beside, as if there
# were one other.  The same bits either way.
@pytest.mark.parametrize("B", [40, 128, 129, 200])
def test_members_have_two_column_tiles_beside_other_streams(B, gpu_device, monkeypatch):
    from rnn_train_ring_attractor_amd import ring_rnn_cuda_func, rnn_cuda, _lib
    monkeypatch.delenv("RINGATTR_TEAM", raising=False)
    N, T = 256, 6
    print(f"[case] rows kernels beside other streams B={B}", flush=True)
    p = make_problem(47, B, T, 2, N)
    t = lambda x: torch.as_tensor(x, dtype=torch.float32, device=gpu_device)
    A, Wa, Wo, r0 = (t(p[n]) for n in ("A", "Wa", "Wo", "r0"))
    long_A = torch.zeros(16, 10000, 2, device=gpu_device)
    long_r = r0[:16].clone()

    def infer():
        with torch.no_grad():
            return ring_rnn_cuda_func(A, Wa, -1.0 / N, 0.5, Wo, r0, 0.15, "gelu"), _lib.last_kernel_names()["fwd"][-4:]

    def train():
        wo = Wo.clone().requires_grad_(True)
        h = ring_rnn_cuda_func(A, Wa, -1.0 / N, 0.5, wo, r0, 0.15, "gelu")
        names = _lib.last_kernel_names()["fwd"][-4:]
        h.backward(torch.ones_like(h))
        return h.detach(), wo.grad, names, _lib.last_kernel_names()["bptt"]

    def beside(streams, call):
        torch.cuda.synchronize()
        for s in streams:
            with torch.cuda.stream(s), torch.no_grad():          # some eight milliseconds each
                ring_rnn_cuda_func(long_A, Wa, -1.0 / N, 0.5, Wo, long_r, 0.15, "gelu")
        out = call()
        torch.cuda.synchronize()
        return out

    others = [torch.cuda.Stream(device=gpu_device) for _ in range(3)]
    alone_i, alone_t = beside([], infer), beside([], train)
    assert alone_i[1] == "1,1>" and alone_t[2] == "1,1>" and alone_t[3].endswith("<false,1>")
    for n in (1, 2, 3):
        one = n == 1 and B <= 128
        got_i, got_t = beside(others[:n], infer), beside(others[:n], train)
        assert got_i[1] == ("1,1>" if one else "1,2>") and got_t[2] == ("1,1>" if one else "1,2>")
        assert got_t[3].endswith("<false,1>" if one else "<false,2>")
        assert torch.equal(got_i[0], alone_i[0]) and torch.equal(got_t[0], alone_t[0]) and torch.equal(got_t[1], alone_t[1])
    again = beside([], infer)
    assert again[1] == "1,1>" and torch.equal(again[0], alone_i[0])

    out = torch.empty_like(alone_i[0])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        rnn_cuda.fwd_cuda.fwd(A=A, Wa=Wa, J0=-1.0 / N, J1=0.5, Wo=Wo, r_init=r0, bump_history=out, alpha=0.15, activation_type=1)
    assert _lib.last_kernel_names()["fwd"][-4:] == ("1,1>" if B <= 128 else "1,2>")
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, alone_i[0])
