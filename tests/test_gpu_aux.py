"""GPU checks of the device-side input generator and of the fused clip + Adam step.

Generator (ringattr_generate_inputs): the reference draws from torch's generator, whose stream no test of the
reference pins; what is fixed is the construction (utils/generate_av_integration_data.py:11-58), so the output is
checked against the structural invariants and closed forms of that construction and against the oracle's bump and
action-signal functions on the generated trials, plus simple distribution checks on large samples.
Optimizer (ringattr_clip_adam): against torch.nn.utils.clip_grad_norm_ + torch.optim.Adam on the CPU, step by step."""
import math

import numpy as np
import pytest
import torch

from oracle import ring_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,k,N,pad,bump", [(64, 120, 2, 120, True, "vm"), (257, 33, 16, 256, True, "gauss"),
                                               (50, 7, 5, 48, False, "gauss"), (4096, 240, 2, 256, True, "vm")],
                         ids=["config0", "k16_padded", "spread", "full_size"])
def test_generated_inputs_follow_the_reference_construction(B, T, k, N, pad, bump, gpu_device):
    from rnn_train_ring_attractor_amd import generate_inputs
    print(f"[case] generator B={B} T={T} k={k} N={N}", flush=True)
    ratios = [0.2, 0.5, 0.8]
    max_av = 0.1 * math.pi
    av, angle, action, r0 = generate_inputs(123, B, T, N, k, zero_ratios_in_rest=ratios, zero_padding=pad, bump=bump)
    av2, angle2, action2, r02 = generate_inputs(123, B, T, N, k, zero_ratios_in_rest=ratios, zero_padding=pad, bump=bump)
    assert all(torch.equal(a, b) for a, b in ((av, av2), (angle, angle2), (action, action2), (r0, r02)))   # a function of the seed
    other = generate_inputs(124, B, T, N, k, zero_ratios_in_rest=ratios, zero_padding=pad, bump=bump)[0]
    assert not torch.equal(av, other)
    av, angle, action, r0 = (x.cpu().numpy().astype(np.float64) for x in (av, angle, action, r0))
    n0 = int(T * 0.1)
    rest = T - n0
    assert np.all(av[:, :n0] == 0.0)
    assert np.abs(av).max() <= max_av
    allowed = {rest - int(np.float32(rest) * np.float32(r)) for r in ratios}
    counts = (av[:, n0:] != 0).sum(axis=1)
    assert set(np.unique(counts)) <= allowed                    # exactly rest - floor(rest * ratio) non-zero steps per trial
    if B >= 64:
        assert set(np.unique(counts)) == allowed                # every ratio is drawn
    assert np.all((angle[:, 0] >= 0) & (angle[:, 0] < 2 * np.pi))
    want = (angle[:, :1] + np.cumsum(av[:, :-1], axis=1)) % (2 * np.pi)
    diff = np.abs(np.angle(np.exp(1j * (angle[:, 1:] - want))))   # compare on the circle (fp32 wrap at 2 pi)
    assert diff.max() <= 1e-4
    assert np.all((angle >= 0) & (angle < 2 * np.pi + 1e-6))
    want_action = O.av_to_action_signal_nd(av, k, zero_padding=pad) if k != 2 or not pad else O.av_to_action_signal(av)
    np.testing.assert_allclose(action, want_action, rtol=1e-6, atol=1e-9)
    want_bump = (O.von_mises_bump if bump == "vm" else O.create_initial_bump)(angle[:, 0], N)
    assert O.max_rel_err(r0, want_bump) <= 1e-5
    np.testing.assert_allclose(np.linalg.norm(r0, axis=1), 1.0, rtol=1e-5)
    if B * rest >= 200_000:
        # distribution: non-zero values are U(-max_av, max_av); positions are chosen uniformly
        vals = av[:, n0:][av[:, n0:] != 0] / max_av
        assert abs(vals.mean()) <= 0.01 and abs(vals.var() - 1.0 / 3.0) <= 0.01
        assert abs(np.mean(np.abs(vals) < 0.5) - 0.5) <= 0.01
        freq = (av[:, n0:] != 0).mean(axis=0)
        assert freq.max() - freq.min() <= 0.06                  # no position favoured (binomial noise ~ 0.008)
        a0 = angle[:, 0] / (2 * np.pi)
        assert abs(a0.mean() - 0.5) <= 0.02 and abs(a0.var() - 1.0 / 12.0) <= 0.01


@pytest.mark.parametrize("T,ratio", [(180, 0.35), (10, 0.7), (120, 0.01)])
def test_generator_leading_zeros_are_pythons_count(T, ratio, gpu_device):
    """int(T * ratio) as Python forms it (a float32 product gives 63 and 6 for the first two pairs instead of 62
    and 7); with a zero ratio of 0 every later step is drawn, so the leading zeros are exactly the count."""
    from rnn_train_ring_attractor_amd import generate_inputs
    print(f"[case] generator leading zeros T={T} ratio={ratio}", flush=True)
    av = generate_inputs(5, 256, T, 64, 2, zero_padding_start_ratio=ratio, zero_ratios_in_rest=[0.0])[0].cpu().numpy()
    n0 = int(T * ratio)
    assert np.all(av[:, :n0] == 0.0)
    assert np.all(av[:, n0:] != 0.0)


def test_generated_inputs_drive_the_operator(gpu_device):
    """Generated tensors go straight into the time loop (zero-padded action channels state the driven ones)."""
    from rnn_train_ring_attractor_amd import generate_inputs, ring_rnn_cuda_func
    B, T, k, N = 64, 30, 8, 256
    av, angle, action, r0 = generate_inputs(5, B, T, N, k)
    gen = torch.Generator(device=gpu_device).manual_seed(1)
    Wa = torch.randn(k, N, N, device=gpu_device, generator=gen) / N ** 0.5
    Wo = torch.randn(N, N, device=gpu_device, generator=gen) / N ** 0.5
    hist = ring_rnn_cuda_func(action, Wa, -0.1, 0.2, Wo, r0, 0.15, "tanh")
    c = lambda t: t.cpu().numpy()
    ref, _ = O.forward_dense(c(action), c(Wa), -0.1, 0.2, c(Wo), c(r0), 0.15, "tanh")
    assert O.max_rel_err(c(hist), ref) <= 1e-2


@pytest.mark.parametrize("max_norm", [1.0, 1e9, 0.0], ids=["clipping", "not_clipping", "clip_off"])
def test_fused_clip_adam_matches_torch(max_norm, gpu_device):
    from rnn_train_ring_attractor_amd import FusedClipAdam
    torch.manual_seed(3)
    shapes = [(256, 256), (2, 256, 256), (16, 1), (16,), (1, 16), (1,), (5000,)]
    ref = [torch.randn(s).requires_grad_(True) for s in shapes]
    dev = [p.detach().clone().to(gpu_device).requires_grad_(True) for p in ref]
    opt_ref = torch.optim.Adam(ref, lr=3e-3, betas=(0.9, 0.99), eps=1e-8)
    opt_dev = FusedClipAdam(dev, lr=3e-3, betas=(0.9, 0.99), eps=1e-8, max_norm=max_norm)
    for step in range(5):
        grads = [torch.randn(s) * (3.0 if step % 2 == 0 else 0.01) for s in shapes]
        for p, q, g in zip(ref, dev, grads):
            p.grad = g.clone()
            q.grad = g.clone().to(gpu_device)
        if max_norm > 0:
            norm = torch.nn.utils.clip_grad_norm_(ref, max_norm)
        else:
            norm = torch.linalg.vector_norm(torch.stack([g.norm() for g in grads]))
        opt_ref.step()
        opt_dev.step()
        torch.cuda.synchronize()
        assert abs(float(opt_dev.last_grad_norm) - float(norm)) <= 1e-5 * float(norm)
        for p, q in zip(ref, dev):
            np.testing.assert_allclose(q.detach().cpu().numpy(), p.detach().numpy(), rtol=2e-5, atol=2e-7)
            np.testing.assert_allclose(q.grad.cpu().numpy(), p.grad.numpy(), rtol=1e-5, atol=1e-9)
    # repeatable bit for bit (fixed summation order of the norm)
    a = [p.detach().clone() for p in dev]
    opt2 = FusedClipAdam([x.clone().requires_grad_(True) for x in a], lr=1e-3, max_norm=0.5)
    opt3 = FusedClipAdam([x.clone().requires_grad_(True) for x in a], lr=1e-3, max_norm=0.5)
    for o in (opt2, opt3):
        for p, g in zip(o.params, grads):
            p.grad = g.clone().to(gpu_device)
        o.step()
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(opt2.params, opt3.params))


# the most partial sums of the norm that every workgroup of the update adds up itself, and one more
@pytest.mark.parametrize("numel", [1024 * 4096, 1024 * 4096 + 1])
def test_fused_clip_adam_of_many_parameters(numel, gpu_device):
    from rnn_train_ring_attractor_amd import FusedClipAdam
    print(f"[case] clip and Adam, {numel} parameters", flush=True)
    w = torch.zeros(numel, device=gpu_device, requires_grad=True)
    w.grad = torch.full((numel,), 0.5, device=gpu_device)
    opt = FusedClipAdam([w], lr=1e-3, betas=(0.9, 0.999), eps=1e-8, max_norm=1.0)
    opt.step()
    torch.cuda.synchronize()
    norm = 0.5 * numel ** 0.5                # sums of 2^-2: exact in fp32 but for the tree's last roundings
    assert abs(float(opt.last_grad_norm) - norm) <= 1e-6 * norm
    g = 0.5 / (norm + 1e-6)
    assert float((w.grad - g).abs().max()) <= 1e-6 * g and float((w.detach() + 1e-3).abs().max()) <= 1e-3 * (1e-5 + 1e-8 / g)


# k a multiple of four and not, a slice that starts off a 16-byte boundary, one sample, more samples than one pass of the grid,
# the most that a single workgroup takes and one more, also with more channels
@pytest.mark.parametrize("B,T,k,N,pair,offset", [(1, 1, 3, 17, (0, 2), 0), (5, 7, 16, 33, (0, 1), 0), (40, 9, 6, 130, (2, 5), 3),
                                                 (700, 513, 4, 20, (1, 3), 1), (8, 128, 16, 33, (0, 1), 0), (25, 41, 16, 33, (0, 1), 0),
                                                 (2, 256, 15, 20, (0, 1), 0), (19, 27, 15, 20, (0, 1), 0), (1, 256, 64, 20, (0, 1), 0),
                                                 (1, 257, 64, 20, (3, 60), 0), (1, 257, 16, 20, (0, 1), 2), (3, 171, 16, 20, (0, 1), 2)])
def test_compacted_channels_are_the_named_ones_and_the_rest_is_checked(B, T, k, N, pair, offset, gpu_device):
    from rnn_train_ring_attractor_amd.ring_rnn_cuda import _compact
    print(f"[case] compaction B={B} T={T} k={k} N={N} {pair}", flush=True)
    A = torch.zeros(B * T * k + offset, device=gpu_device)[offset:].view(B, T, k)
    for c in pair:
        A[..., c] = torch.randn(B, T, device=gpu_device)
    Wa = torch.randn(k, N, N, device=gpu_device)
    a2, w2 = _compact(A, Wa, pair)
    assert torch.equal(a2, A[..., list(pair)]) and torch.equal(w2, Wa[list(pair)])
    silent = [c for c in range(k) if c not in pair]
    for b, t, c, v in ((B - 1, T - 1, silent[-1], 1e-30), (0, 0, silent[0], float("nan"))):
        A[b, t, c] = v
        assert torch.isnan(_compact(A, Wa, pair)[0]).all()
        A[b, t, c] = 0.0


@pytest.mark.parametrize("N,k", [(60, 16), (300, 5), (600, 6)])
def test_a_padded_signal_that_was_written_to_gives_its_own_results(N, k, gpu_device):
    """Outside the weight-resident widths the helper's statement decides nothing: a silent channel that has been written to
    counts, also where the tensor's version counter has not seen the write."""
    from rnn_train_ring_attractor_amd import host, ring_rnn_cuda_func
    from rnn_train_ring_attractor_amd.ring_rnn_cuda import _driven_pair
    B, T = 20, 6
    print(f"[case] padded signal N={N} k={k}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(3)
    r = lambda *s: torch.randn(*s, device=gpu_device, generator=g)
    A, r0, G = host.av_to_action_signal_ND(r(B, T) * 0.2, k), r(B, N).abs() * 0.1, r(T, B, N)
    wa, wo, outs = r(k, N, N) / N ** 0.5, r(N, N) / N ** 0.5, []
    for signal in (A, A.clone()):                      # (a copy carries no statement)
        Wa, Wo = wa.clone().requires_grad_(True), wo.clone().requires_grad_(True)
        h = ring_rnn_cuda_func(signal, Wa, -0.05, 0.5, Wo, r0, 0.15, "tanh")
        h.backward(G)
        outs.append((h.detach(), Wa.grad, Wo.grad))
    assert _driven_pair(A, Wa) is None and _driven_pair(A.clone(), Wa) is None
    assert torch.count_nonzero(outs[0][1][2:]) == 0
    for x, y in zip(*outs):
        assert torch.equal(x, y)
    A.data[0, 0, 2] = 0.1
    for _ in range(2):
        want = ring_rnn_cuda_func(A.clone(), Wa, -0.05, 0.5, Wo, r0, 0.15, "tanh")
        assert torch.isfinite(want).all() and torch.equal(ring_rnn_cuda_func(A, Wa, -0.05, 0.5, Wo, r0, 0.15, "tanh"), want)
        A[0, 0, 2] = 0.2


@pytest.mark.parametrize("B,T,k", [(1, 1, 2), (5, 7, 3), (33, 20, 16), (700, 513, 5)])
def test_action_signal_in_one_launch_equals_the_tensor_operations(B, T, k, gpu_device):
    from rnn_train_ring_attractor_amd import host
    print(f"[case] action signal B={B} T={T} k={k}", flush=True)
    av = torch.randn(B, T, device=gpu_device)
    av[0, 0] = float("nan")
    av[-1, -1] = 0.0
    for fast, slow in ((host.av_to_action_signal_ND(av, k), host.av_to_action_signal_ND(av.clone().requires_grad_(True), k)),
                       (host.av_to_action_signal(av), host.av_to_action_signal(av.cpu()).to(gpu_device))):
        assert fast.shape == slow.shape and torch.equal(torch.nan_to_num(fast, 7.0), torch.nan_to_num(slow.detach(), 7.0))


@pytest.mark.parametrize("B,N,width", [(1, 1, 10), (3, 17, 10), (130, 256, 7.5), (9, 2048, 10)])
def test_initial_bump_in_one_launch_equals_the_tensor_operations(B, N, width, gpu_device):
    from rnn_train_ring_attractor_amd import host
    print(f"[case] initial bump B={B} N={N}", flush=True)
    angle = torch.rand(B, 5, device=gpu_device, dtype=torch.float32) * 6.283
    angle[0, 0] = 0.0
    got = host.create_initial_bump(angle[:, 0], N, width, device=gpu_device)
    want = host.create_initial_bump(angle[:, 0].clone().requires_grad_(True), N, width, device=gpu_device)
    assert want.requires_grad and not got.requires_grad and torch.equal(got, want.detach())      # the same roundings


def test_helpers_keep_to_tensor_operations_where_something_watches_them(gpu_device):
    """vmap, forward mode and tracing see the operations themselves."""
    from rnn_train_ring_attractor_amd import host
    av = torch.randn(3, 4, 5, device=gpu_device)
    assert torch.equal(torch.func.vmap(host.av_to_action_signal)(av), torch.stack([host.av_to_action_signal(a) for a in av]))
    angle = torch.rand(4, device=gpu_device)
    _, tangent = torch.func.jvp(lambda a: host.create_initial_bump(a, 32, device=gpu_device), (angle,), (torch.ones_like(angle),))
    assert float(tangent.abs().max()) > 0
    traced = torch.jit.trace(lambda a: host.av_to_action_signal(a), av[0])
    assert torch.equal(traced(av[1]), host.av_to_action_signal(av[1]))


@pytest.mark.parametrize("owner,name", [("torch._C._functorch", "maybe_current_level"), ("torch.autograd.forward_ad", "_current_level"),
                                        ("torch._C", "_len_torch_dispatch_stack"), ("torch._C", "_len_torch_function_stack")])
def test_helpers_keep_to_tensor_operations_where_torch_lacks_a_private_name(owner, name, gpu_device, monkeypatch):
    import operator
    from rnn_train_ring_attractor_amd import _lib, host
    av, angle = torch.randn(4, 5, device=gpu_device), torch.rand(4, device=gpu_device)
    want = host.av_to_action_signal(av), host.av_to_action_signal_ND(av, 5), host.create_initial_bump(angle, 32, device=gpu_device)
    assert _lib.plain_gpu_tensor(av)
    monkeypatch.delattr(operator.attrgetter(owner.partition(".")[2])(torch), name)
    assert not _lib.plain_gpu_tensor(av)
    got = host.av_to_action_signal(av), host.av_to_action_signal_ND(av, 5), host.create_initial_bump(angle, 32, device=gpu_device)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_stream_handle_is_the_current_streams(gpu_device, monkeypatch):
    from rnn_train_ring_attractor_amd import _lib
    side = torch.cuda.Stream()
    device = torch.zeros(1, device=gpu_device).device
    for missing in (False, True):                      # (torch's private name may be missing)
        if missing:
            monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
        assert _lib.stream_handle(device) == torch.cuda.current_stream(device).cuda_stream
        with torch.cuda.stream(side), _lib.on_device(device):
            assert _lib.stream_handle(device) == side.cuda_stream and torch.cuda.current_device() == device.index
