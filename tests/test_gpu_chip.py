"""GPU tests of the chip kernels (forward without a record of wide rings, the weights on chip across all compute units):
the fp64 oracle, the same bits whatever the members' width, from single workgroups where a row group does not gather, in any
batch and in replayed graphs, and the rule that takes calls there."""
import numpy as np
import pytest
import torch

from oracle import ring_oracle as O
from tests.ring_cases import make_problem

pytestmark = pytest.mark.gpu

SWITCHES = ("RINGATTR_CHIP", "RINGATTR_TEAM", "RINGATTR_TEAM_GATHER_US", "RINGATTR_PANEL", "RINGATTR_PANEL_SHAPE", "RINGATTR_BLOCK", "RINGATTR_WIDE",
            "RINGATTR_BLOCK_SHAPE", "RINGATTR_STREAMING", "RINGATTR_CLUSTER")


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in SWITCHES:
        monkeypatch.delenv(name, raising=False)


def _tensors(p, dev):
    return [torch.as_tensor(p[x], dtype=torch.float32, device=dev) for x in ("A", "Wa", "Wo", "r0")]


def _forward(t, act, J0, J1):
    from rnn_train_ring_attractor_amd import _lib, ring_rnn_cuda_func
    A, Wa, Wo, r0 = t
    with torch.no_grad():
        h = ring_rnn_cuda_func(A, Wa, J0, J1, Wo, r0, 0.15, act)
    return h, _lib.last_kernel_names()["fwd"]


# rows: one, a whole tile, ragged, one to many tiles per row group, more groups than tiles; neurons: the fewest, K chunks that
# are not whole, one past a wave's share of them (769, 1025, 1537), no multiple of four, the most; channels: one, an even and
# an odd number of matrices, more than fit the registers, sixteen, a silent one; more steps than slots
@pytest.mark.parametrize("B,T,k,N,act", [
    (1, 3, 7, 513, "relu"), (9, 3, 1, 1200, "tanh"), (16, 12, 5, 640, "gelu"), (100, 6, 16, 700, "silu"), (33, 9, 6, 769, "tanh"), (7, 2, 12, 1023, "gelu"),
    (40, 10, 16, 1024, "tanh"), (300, 5, 3, 1025, "gelu"), (50, 4, 2, 1300, "silu"), (20, 9, 16, 1536, "gelu"), (130, 3, 7, 1537, "relu"),
    (17, 1, 2, 2047, "tanh"), (64, 9, 13, 2048, "silu"), (1, 20, 3, 2048, "gelu"),
])
def test_chip_kernels_against_the_oracle(B, T, k, N, act, gpu_device, monkeypatch):
    print(f"[case] chip B={B} T={T} k={k} N={N} {act}", flush=True)
    J0, J1 = -1.0 / N, 0.5
    p = make_problem(11, B, T, k, N, bump="vm", action="dense")
    if k > 2:
        p["A"][:, :, 1] = 0.0
    t = _tensors(p, gpu_device)
    ref, _ = O.forward_dense(p["A"], p["Wa"], J0, J1, p["Wo"], p["r0"], 0.15, act)
    ran = {}
    for width in ("1", "8", "16", "32"):                 # (1: the rule's own choice)
        monkeypatch.setenv("RINGATTR_CHIP", width)
        h, name = _forward(t, act, J0, J1)
        if "chip" in name:
            ran[width] = h
    assert "1" in ran and len(ran) >= 2                  # not every width has room for every number of channels
    got = ran["1"]
    assert O.max_rel_err(got.cpu().numpy(), ref) <= 1e-2 # one bf16 rounding per operand, as everywhere
    assert all(torch.equal(got, h) for h in ran.values())
    monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")  # no group gathers: a workgroup per tile
    for width in ran:
        monkeypatch.setenv("RINGATTR_CHIP", width)
        h, _ = _forward(t, act, J0, J1)
        assert torch.equal(got, h)
    monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
    monkeypatch.setenv("RINGATTR_CHIP", "1")
    rows = slice(B // 2, B)                              # the same rows in another batch
    h, name = _forward([t[0][rows].clone(), t[1], t[2], t[3][rows].clone()], act, J0, J1)
    assert "chip" in name and torch.equal(h, got[:, rows])


def test_infinite_states_and_absent_matrices(gpu_device, monkeypatch):
    """Column tiles hold an even number of matrices; the one that is not there takes nothing from an infinite state."""
    monkeypatch.setenv("RINGATTR_CHIP", "8")
    B, T, k, N = 5, 4, 2, 1100
    p = make_problem(12, B, T, k, N, bump="vm", action="dense")
    p["Wo"], p["Wa"] = np.abs(p["Wo"]), np.abs(p["Wa"])
    p["A"] = np.abs(p["A"]) + 0.1
    p["r0"][2] = np.inf
    h, name = _forward(_tensors(p, gpu_device), "relu", 0.0, 1.0)
    assert "chip" in name
    assert torch.isinf(h[:, 2]).all() and torch.isfinite(h[:, [0, 1, 3, 4]]).all()


# one, two, three and more tiles per row group (8, 6, 6 and 4 slots), operands one to three items ahead, one to eight row groups, the
# last of them a tile short
@pytest.mark.parametrize("B,k,N,width", [
    (16, 3, 1100, "8"), (32, 3, 1100, "16"), (64, 3, 1100, "16"), (41, 8, 1100, "8"), (41, 16, 1100, "8"), (73, 7, 600, "8"), (100, 16, 1024, "8"),
    (120, 10, 900, "8"), (300, 3, 1021, "32"), (400, 4, 900, "16"), (150, 2, 2048, "32"), (256, 2, 2048, "32")])
def test_slots_come_round_many_times(B, k, N, width, gpu_device, monkeypatch):
    """150 steps, 19 to 37 rounds through the exchange slots: every row has the bits that the way without slots gives it."""
    print(f"[case] chip rounds B={B} k={k} N={N} width {width}", flush=True)
    t = _tensors(make_problem(13, B, 150, k, N, bump="vm", action="dense"), gpu_device)
    monkeypatch.setenv("RINGATTR_CHIP", width)
    h, name = _forward(t, "tanh", -1.0 / N, 0.9)
    assert "chip" in name
    monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")
    without, _ = _forward(t, "tanh", -1.0 / N, 0.9)
    assert torch.equal(without, h)
    monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
    if N > 1024 or k > 3:                                # the same rows a few at a time: other numbers of tiles and slots
        monkeypatch.setenv("RINGATTR_CHIP", "8")         # (nine rows of N <= 1024 and three channels are the teams')
        part, name = _forward([t[0][:9].clone(), t[1], t[2], t[3][:9].clone()], "tanh", -1.0 / N, 0.9)
        assert "chip" in name and torch.equal(part, h[:, :9])


# Every kernel that is built, but for those of FEW_CHANNELS: neurons per workgroup, K chunks and column tiles of a wave, the fewest and the
# most channels that take that many column tiles, and how many operands can be on their way at most.
KERNELS = [
    (8, 3, 4, 5, 7, 3), (8, 3, 7, 8, 13, 3), (8, 3, 9, 14, 16, 3), (8, 4, 4, 4, 7, 3), (8, 4, 7, 8, 13, 3), (8, 4, 9, 14, 16, 3),
    (8, 6, 2, 1, 3, 3), (8, 6, 4, 4, 7, 3), (8, 6, 7, 8, 13, 2), (8, 6, 9, 14, 16, 1), (8, 8, 2, 1, 3, 3), (8, 8, 4, 4, 7, 2), (8, 8, 7, 8, 13, 1),
    (16, 3, 7, 5, 6, 3), (16, 4, 7, 4, 6, 3), (16, 6, 3, 1, 2, 3), (16, 6, 4, 3, 3, 3), (16, 6, 7, 4, 6, 2), (16, 8, 3, 1, 2, 2), (16, 8, 4, 3, 3, 2),
    (16, 8, 7, 4, 6, 1), (32, 6, 6, 1, 2, 2), (32, 6, 8, 3, 3, 2), (32, 8, 6, 1, 2, 1),
]
# Up to three channels at N <= 1024 come here with many rows only (the teams take the others): workgroup, chunks, tiles, operands on
# their way, N, channels, rows
FEW_CHANNELS = [
    (8, 3, 2, 3, 765, 3, 2317), (8, 4, 2, 3, 1001, 3, 265), (8, 4, 2, 3, 1024, 3, 400), (16, 3, 4, 3, 517, 3, 2957), (16, 4, 3, 3, 779, 1, 3117),
    (16, 4, 4, 3, 1021, 3, 265), (32, 3, 6, 3, 513, 1, 4557), (32, 3, 6, 3, 768, 2, 4557), (32, 3, 8, 3, 516, 3, 2957), (32, 4, 6, 3, 778, 1, 3117),
    (32, 4, 8, 2, 1021, 3, 378), (32, 4, 8, 2, 1024, 3, 265), (32, 4, 8, 3, 1021, 3, 633)]
WIDTHS = {3: (517, 764), 4: (771, 1024), 6: (1031, 1536), 8: (1541, 2048)}           # N by K chunks of a wave: odd, a multiple of four


@pytest.mark.parametrize("npw,kpw,ct,fewest,most,depth", KERNELS)
def test_every_kernel(npw, kpw, ct, fewest, most, depth, gpu_device, monkeypatch):
    """One to five tiles per row group, the last group's one short: the oracle for rows of the first, a middle and the last tile, every
    row the bits of the way without slots and of every other batch.  With one or two tiles an operand is asked for behind the item
    before, with three one item ahead, two only where every group has four."""
    T = 12
    for N, k in zip(WIDTHS[kpw], (fewest, most)):
        groups = 8
        while 32 * ((N + 31) // 32) // npw > 256 // groups:
            groups //= 2
        batches = [16 * groups - 7] + [16 * (groups * (nt - 1) + max(1, groups - 1)) - 7 for nt in (2, 3, 4, 5)]
        batches = batches[:2] if (npw, kpw, ct) == (16, 8, 7) else batches           # (LDS holds two tiles' states beside its weights)
        print(f"[case] chip <{npw}, {kpw}, {ct}> N={N} k={k} B={batches}", flush=True)
        J0, J1, B = -1.0 / N, 0.6, batches[-1]
        p = make_problem(19 + ct, B, T, k, N, bump="vm", action="dense")
        t = _tensors(p, gpu_device)
        monkeypatch.setenv("RINGATTR_CHIP", str(npw))
        monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")
        want, _ = _forward(t, "gelu", J0, J1)
        monkeypatch.delenv("RINGATTR_TEAM_GATHER_US")
        for nt, rows in enumerate(batches, 1):
            h, name = _forward([t[0][:rows].clone(), t[1], t[2], t[3][:rows].clone()], "gelu", J0, J1)
            ahead = 1 if nt <= 2 else 3 if (rows + 15) // 16 // groups >= 4 else 2
            assert f"<{npw},{kpw},{ct},{min(ahead, depth)}>" in name, (N, k, rows, name)
            assert torch.equal(h, want[:, :rows]), (N, k, rows)
        some = [0, 15, B // 2, B - 1]
        ref, _ = O.forward_dense(p["A"][some], p["Wa"], J0, J1, p["Wo"], p["r0"][some], 0.15, "gelu")
        assert O.max_rel_err(want[:, some].cpu().numpy(), ref) <= 1e-2               # one bf16 rounding per operand, as everywhere


@pytest.mark.parametrize("npw,kpw,ct,depth,N,k,B", FEW_CHANNELS)
def test_every_kernel_of_few_channels(npw, kpw, ct, depth, N, k, B, gpu_device, monkeypatch):
    print(f"[case] chip <{npw}, {kpw}, {ct}, {depth}> N={N} k={k} B={B}", flush=True)
    J0, J1 = -1.0 / N, 0.6
    p = make_problem(23, B, 12, k, N, bump="vm", action="dense")
    t = _tensors(p, gpu_device)
    monkeypatch.setenv("RINGATTR_CHIP", str(npw))
    h, name = _forward(t, "silu", J0, J1)
    assert f"<{npw},{kpw},{ct},{depth}>" in name, name
    monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "-1")
    without, _ = _forward(t, "silu", J0, J1)
    assert torch.equal(h, without)
    some = [0, 15, B // 2, B - 1]
    ref, _ = O.forward_dense(p["A"][some], p["Wa"], J0, J1, p["Wo"], p["r0"][some], 0.15, "silu")
    assert O.max_rel_err(h[:, some].cpu().numpy(), ref) <= 1e-2                      # one bf16 rounding per operand, as everywhere


def test_replayed_graph(gpu_device):
    B, T, k, N = 20, 12, 6, 1024
    t = _tensors(make_problem(14, B, T, k, N, bump="vm", action="dense"), gpu_device)
    want, name = _forward(t, "gelu", -1.0 / N, 0.9)
    assert "chip" in name
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _forward(t, "gelu", -1.0 / N, 0.9)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out, _ = _forward(t, "gelu", -1.0 / N, 0.9)
    torch.cuda.current_stream().wait_stream(side)
    scale = 1.0
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        scale *= 0.5
        t[3].mul_(scale)
        want, _ = _forward(t, "gelu", -1.0 / N, 0.9)


# Where the default takes a call: few steps, two channels that the teams take, narrow rings, more channels than are built, more weights than fit
# (17 matrices past N = 1536), batches that take longer than on the panels, and those that would if only two channels were driven
@pytest.mark.parametrize("B,T,k,N,chip", [
    (1, 12, 6, 1024, True), (64, 12, 2, 1100, True), (256, 12, 6, 1024, True), (1, 12, 13, 2048, True),
    (1, 9, 6, 1024, False), (1, 12, 2, 1024, False), (1, 12, 6, 512, False), (1, 12, 17, 1100, False), (256, 12, 16, 2048, False), (1, 12, 14, 2048, False),
    (1024, 10, 2, 2048, False), (1024, 10, 16, 1024, False), (64, 12, 16, 1500, False), (256, 12, 16, 1024, False), (1024, 10, 6, 640, False)])
def test_rule(B, T, k, N, chip, gpu_device):
    _, name = _forward(_tensors(make_problem(15, B, T, k, N, bump="vm", action="dense"), gpu_device), "relu", 0.0, 0.5)
    assert ("chip" in name) == chip, name


# two of the channels driven; three tiles in every row group, and four in all but one
@pytest.mark.parametrize("B,k,N", [(89, 16, 896), (107, 8, 891), (75, 14, 920)])
def test_few_tiles_per_group_take_no_longer_than_the_panels(B, k, N, gpu_device, monkeypatch):
    """An operand that was asked for before it could be there held up what it waited for (896: 404 us, the panels 331; now 239)."""
    T = 40
    p = make_problem(20, B, T, k, N, bump="vm", action="dense")
    p["A"][:, :, 2:] = 0.0
    t = _tensors(p, gpu_device)
    least = {}
    for switch, want in (("", "chip"), ("0", "panel"), ("", "chip"), ("0", "panel")):
        if switch:
            monkeypatch.setenv("RINGATTR_CHIP", switch)
        else:
            monkeypatch.delenv("RINGATTR_CHIP", raising=False)
        for _ in range(6):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            _, name = _forward(t, "tanh", -1.0 / N, 0.5)
            end.record()
            torch.cuda.synchronize()
            assert want in name
            least[want] = min(least.get(want, 1e9), start.elapsed_time(end))
    print(f"[case] B={B} k={k} N={N}: chip {least['chip']:.3f} ms, panels {least['panel']:.3f}", flush=True)
    assert least["chip"] < least["panel"]


def test_row_groups_that_do_not_gather_cost_little(gpu_device, monkeypatch):
    """Compute units held by another stream, graph or process: the tiles are done on those there are, in a small multiple of the panel
    kernels' time (a workgroup per tile took nearly a thousand times as long)."""
    B, T, k, N = 1, 12, 12, 2048
    t = _tensors(make_problem(16, B, T, k, N, bump="vm", action="dense"), gpu_device)

    def ms(want, **switches):
        for name, value in switches.items():
            monkeypatch.setenv(name, value)
        times = []
        for _ in range(3):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            h, kernel = _forward(t, "gelu", -1.0 / N, 0.5)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
            assert want in kernel
        for name in switches:
            monkeypatch.delenv(name)
        return min(times), h

    _, whole = ms("chip")
    rest, h = ms("chip", RINGATTR_TEAM_GATHER_US="-1")
    panel, _ = ms("panel", RINGATTR_CHIP="0")
    print(f"[case] chip, no group gathered: {rest:.2f} ms, panels {panel:.2f} ms", flush=True)
    assert torch.equal(h, whole) and rest < 20 * panel


# all row groups, and those that are not complete at once; one and several row groups, tile blocks that are not full
@pytest.mark.parametrize("B,T,k,N", [(1, 12, 6, 1024), (100, 10, 16, 700), (378, 10, 3, 1021), (130, 11, 2, 1537), (250, 10, 5, 640)])
def test_groups_that_are_not_complete_in_time(B, T, k, N, gpu_device, monkeypatch):
    print(f"[case] chip groups give up B={B} T={T} k={k} N={N}", flush=True)
    monkeypatch.setenv("RINGATTR_CHIP", "1")
    monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", "1000000")
    t = _tensors(make_problem(17, B, T, k, N, bump="vm", action="dense"), gpu_device)
    want, name = _forward(t, "silu", -1.0 / N, 0.8)
    assert "chip" in name
    for wait_us in ("-1", "0", "2", "10"):
        monkeypatch.setenv("RINGATTR_TEAM_GATHER_US", wait_us)
        for _ in range(2):
            h, _ = _forward(t, "silu", -1.0 / N, 0.8)
            assert torch.equal(h, want), wait_us


@pytest.mark.parametrize("B,T,k,N", [(40, 12, 6, 1024), (20, 10, 2, 2000)])
def test_two_streams_and_two_graphs(B, T, k, N, gpu_device, monkeypatch):
    """Launches that each want every compute unit: eager ones are ordered by the library, replayed graphs are not."""
    monkeypatch.setenv("RINGATTR_CHIP", "1")
    t = _tensors(make_problem(18, B, T, k, N, bump="vm", action="dense"), gpu_device)
    want, name = _forward(t, "tanh", -1.0 / N, 0.9)
    assert "chip" in name
    print("[case] chip on two streams", flush=True)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for _ in range(3):
        for s in streams:
            with torch.cuda.stream(s):
                got.append(_forward(t, "tanh", -1.0 / N, 0.9)[0])
    torch.cuda.synchronize()
    assert all(torch.equal(h, want) for h in got)
    graphs, outs = [], []
    for s in streams:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            outs.append(_forward(t, "tanh", -1.0 / N, 0.9)[0])
        graphs.append(graph)
    for _ in range(4):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        print("[case] chip graphs on two streams", flush=True)
        for s, graph in zip(streams, graphs):
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o in outs)
    _forward(t, "tanh", -1.0 / N, 0.9)          # (a wait that had run out would be reported by this call)
