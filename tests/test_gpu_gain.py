"""GPU parity of the gain-network operator (ringattr_gain_fwd / ringattr_gain_bwd through the Python operator and
the C ABI) against the fp64 oracle, which is itself pinned to the reference's nn.Sequential construction."""
import numpy as np
import pytest
import torch

from oracle import ring_oracle as O

pytestmark = pytest.mark.gpu


def _case(seed, B, T, k, h, signed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((B, T, k)).astype(np.float32) * 0.3
    if not signed:
        x = np.maximum(x, 0.0)                                # the (L, R) channels are rectified
    params = (rng.standard_normal((k, 3 * h + 1)) / np.sqrt(h)).astype(np.float32)
    g = rng.standard_normal((B, T, k)).astype(np.float32)
    return x, params, g


@pytest.mark.parametrize("B,T,k,h,signed", [(64, 120, 2, 16, False), (37, 9, 3, 16, True), (5, 3, 1, 4, True),
                                            (128, 33, 16, 8, True), (21, 7, 2, 32, False), (19, 5, 4, 20, True)],
                         ids=["lr_h16", "ragged_k3", "tiny_h4", "k16_h8", "h32", "h20_padded"])
def test_gain_operator_matches_oracle(B, T, k, h, signed, gpu_device):
    from rnn_train_ring_attractor_amd import ring_gain_func
    print(f"[case] gain B={B} T={T} k={k} h={h}", flush=True)
    x, params, g = _case(7, B, T, k, h, signed)
    xt = torch.tensor(x, device=gpu_device, requires_grad=True)
    pt = torch.tensor(params, device=gpu_device, requires_grad=True)
    out = ring_gain_func(xt, pt)
    out.backward(torch.tensor(g, device=gpu_device))
    torch.cuda.synchronize()
    ref = O.gain_forward(x, params)
    gp, gx = O.gain_backward(x, params, g)
    # fp32 arithmetic against fp64: relative to the largest magnitude
    assert O.max_rel_err(out.detach().cpu().numpy(), ref) <= 1e-5
    assert O.max_rel_err(pt.grad.cpu().numpy(), gp) <= 1e-4
    assert O.max_rel_err(xt.grad.cpu().numpy(), gx) <= 1e-5
    assert O.cosine(pt.grad.cpu().numpy(), gp) >= 0.999999


def test_gain_gradients_are_repeatable_and_additive_at_full_size(gpu_device):
    """B*T of the gain-network benchmark shape (4096 x 240 samples, two channels): bitwise repeatable parameter
    gradients; two half-batch shards add up to the full batch; a slice agrees with the oracle."""
    from rnn_train_ring_attractor_amd import ring_gain_func
    B, T, k, h = 4096, 240, 2, 16
    gen = torch.Generator(device=gpu_device).manual_seed(11)
    x = torch.relu(torch.randn(B, T, k, device=gpu_device, generator=gen) * 0.2)
    params = torch.randn(k, 3 * h + 1, device=gpu_device, generator=gen) / h ** 0.5
    g = torch.randn(B, T, k, device=gpu_device, generator=gen)

    def run(rows):
        p = params.clone().requires_grad_(True)
        out = ring_gain_func(x[rows].contiguous(), p)
        out.backward(g[rows].contiguous())
        return out.detach(), p.grad

    full, again = run(slice(0, B)), run(slice(0, B))
    assert torch.equal(full[0], again[0]) and torch.equal(full[1], again[1])
    lo, hi = run(slice(0, B // 2)), run(slice(B // 2, B))
    assert O.max_rel_err((lo[1] + hi[1]).cpu().numpy(), full[1].cpu().numpy()) <= 1e-5
    sl = slice(100, 164)
    part = run(sl)
    c = lambda t: t.cpu().numpy()
    assert O.max_rel_err(c(part[0]), O.gain_forward(c(x[sl]), c(params))) <= 1e-5
    gp, _ = O.gain_backward(c(x[sl]), c(params), c(g[sl]))
    assert O.max_rel_err(c(part[1]), gp) <= 1e-4


@pytest.mark.parametrize("B,T,h,k", [(1, 1, 1, 1), (7, 5, 3, 2), (300, 40, 16, 2), (20, 9, 32, 16)])
def test_networks_read_in_place_equal_the_packed_operator(B, T, h, k, gpu_device):
    """Same kernels, parameters by pointer: the same bits, forward and every parameter's gradient; the angular velocity's
    halves likewise."""
    from rnn_train_ring_attractor_amd import gain
    print(f"[case] gain networks in place B={B} T={T} h={h} k={k}", flush=True)
    torch.manual_seed(2)
    nets = [torch.nn.Sequential(torch.nn.Linear(1, h), torch.nn.GELU(), torch.nn.Linear(h, 1), torch.nn.Softplus()).to(gpu_device)
            for _ in range(k)]
    params = [p for net in nets for p in net.parameters()]

    def grads(out, g):
        return [out.detach()] + list(torch.autograd.grad(out, params, g))

    x, av = torch.randn(B, T, k, device=gpu_device), torch.randn(B, T, device=gpu_device)
    g = torch.randn(B, T, k, device=gpu_device)
    for a, b in zip(grads(gain.ring_gain_nets(x, nets), g), grads(gain.ring_gain_func(x, gain.pack_gain_nets(nets)), g)):
        assert a.shape == b.shape and torch.equal(a, b)
    if k == 2:
        base = torch.stack([torch.relu(-av), torch.relu(av)], dim=2)
        for a, b in zip(grads(gain.ring_gain_halves(av, nets), g), grads(gain.ring_gain_func(base, gain.pack_gain_nets(nets)), g)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("write", ["in_place", "data", "adam"])
def test_networks_and_velocity_may_be_written_to_before_the_backward(write, gpu_device):
    """Gradients are those of the values the forward saw, as with the packed operator, which works on new tensors."""
    from rnn_train_ring_attractor_amd import FusedClipAdam, gain
    B, T, h = 33, 21, 5
    print(f"[case] gain networks written to before the backward: {write}", flush=True)
    g = torch.randn(B, T, 2, device=gpu_device)
    av0 = torch.randn(B, T, device=gpu_device)
    grads = []
    for fused in (True, False):
        torch.manual_seed(4)
        nets = [torch.nn.Sequential(torch.nn.Linear(1, h), torch.nn.GELU(), torch.nn.Linear(h, 1), torch.nn.Softplus()).to(gpu_device)
                for _ in range(2)]
        params = [p for net in nets for p in net.parameters()]
        av = av0.clone()
        base = lambda: torch.stack([torch.relu(-av), torch.relu(av)], dim=2)
        x = base()
        outs = [gain.ring_gain_halves(av, nets), gain.ring_gain_nets(x, nets)] if fused else \
               [gain.ring_gain_func(base(), gain.pack_gain_nets(nets)), gain.ring_gain_func(x, gain.pack_gain_nets(nets))]
        if write == "adam":
            for p in params:
                p.grad = torch.ones_like(p)
            FusedClipAdam(params, lr=0.5, max_norm=0.0).step()
        with torch.no_grad():
            for p in params:
                if write == "in_place":
                    p.add_(1.0)
                elif write == "data":
                    p.data.mul_(-2.0)
            (av if write == "in_place" else av.data).fill_(0.3)
        grads.append([t for out in outs for t in torch.autograd.grad(out, params, g)])
    for a, b in zip(*grads):
        assert torch.equal(a, b)
