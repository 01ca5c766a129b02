"""The LAMB kernels against the element-wise operations and against the same
step in 64 bits: tensor sizes at the edges of a workgroup's 4096 elements and of
a 16-byte access, unaligned views, zero norms, more tensors than one launch
takes, and lists that have to take the element-wise way."""

import pytest
import torch

from orion_amd import kernels
from orion_amd.benchmark_suite.transformer_xl import Lamb

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _optimizer(sizes, offset, decay, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    params = []
    for i, n in enumerate(sizes):
        def make(scale):
            flat = torch.empty(n + offset, device=DEV).normal_(0.0, scale, generator=g)
            return flat[offset:]
        p = torch.nn.Parameter(make(0.0 if i == 1 else 1.0))
        p.grad = make(1e-3)
        params.append(p)
    opt = Lamb(params, lr=0.1, weight_decay=decay)
    for p in params:
        opt.state[p]["m"] = torch.empty_like(p).normal_(0.0, 1e-3, generator=g)
        opt.state[p]["v"] = torch.empty_like(p).normal_(0.0, 1e-6, generator=g).abs_()
    return opt, params


def _step64(opt, params):
    out = []
    group = opt.param_groups[0]
    for p in params:
        w, g = p.detach().double(), p.grad.double()
        m, v = opt.state[p]["m"].double(), opt.state[p]["v"].double()
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        u = m / (v.sqrt() + 1e-6) + group["weight_decay"] * w
        wn, un = w.norm().clamp(0, 10), u.norm()
        ratio = 1.0 if wn == 0 or un == 0 else wn / (un + 1e-6)
        out.append((w - 0.1 * ratio * u, m, v))
    return out


@pytest.mark.parametrize("decay", [0.0, 0.01])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("sizes", [(1, 5, 4095, 4096, 4097, 8192), (3, 0, 70001),
                                   tuple(range(1, 140)), ((1 << 26) + 5, 4096, 1 << 20)])
def test_step_against_64_bits(sizes, offset, decay):
    opt, params = _optimizer(sizes, offset, decay)
    assert kernels.lamb_takes(params, [p.grad for p in params], *(
        [opt.state[p][k] for p in params] for k in "mv"))
    want = _step64(opt, params)
    versions = [p._version for p in params]
    opt.step()
    for p, old, (w, m, v) in zip(params, versions, want):
        assert p._version > old
        for got, ref in ((p, w), (opt.state[p]["m"], m), (opt.state[p]["v"], v)):
            # a dozen fp32 roundings of 6e-8 each, the ratio's among them
            assert torch.allclose(got.detach().double(), ref, rtol=1e-6,
                                  atol=1e-6 * float(ref.abs().max()) if ref.numel() else 0)


@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("sizes", [
    # the last complete window of eight workgroups' 4096 elements, and what lies behind it
    (32767, 32768, 32769, 36864, 65535, 65537, 98304 + 4095),
    # every place of a tensor among the 64 of a launch, some of several workgroups
    tuple(1 + 4099 * (i % 7) for i in range(129))])
def test_windows_and_the_tensor_of_a_workgroup(sizes, offset):
    test_step_against_64_bits(sizes, offset, 0.01)


def test_same_bits_twice():
    runs = []
    for _ in range(2):
        opt, params = _optimizer((1 << 20, 77, 300001), 0, 0.01, seed=4)
        opt.step()
        runs.append([p.detach().clone() for p in params])
    assert all(torch.equal(a, b) for a, b in zip(*runs))


def test_infinite_and_nan_gradients_reach_the_weights_as_before():
    for bad in (float("inf"), float("nan")):
        results = []
        for dense in (True, False):
            opt, params = _optimizer((4096, 64, 5000), 0, 0.0, seed=5)
            params[0].grad[7] = bad
            if not dense:          # the element-wise way
                opt.param_groups[0]["lr"] = torch.tensor(0.1, device=DEV)
            opt.step()
            results.append([p.detach().isnan() for p in params])
        assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan")])
@pytest.mark.parametrize("decay", [0.0, 0.01])
def test_infinite_and_nan_weights_give_what_the_operations_give(decay, bad):
    results = []
    for dense in (True, False):
        opt, params = _optimizer((8, 64, 5000), 0, decay, seed=6)
        params[0].data[3] = bad             # a workgroup's part of a chunk
        params[2].data[100] = bad           # a whole one
        if not dense:          # the element-wise way
            opt.param_groups[0]["lr"] = torch.tensor(0.1, device=DEV)
        opt.step()
        results.append([p.detach().clone() for p in params])
    for got, want in zip(*results):
        # a dozen fp32 roundings of 6e-8 each on either side
        finite = want[want.isfinite()]
        top = float(finite.abs().max()) if finite.numel() else 0.0
        assert torch.allclose(got, want, rtol=2e-6, atol=2e-6 * top, equal_nan=True)
    if decay == 0.0 and bad == bad:
        # without decay an infinite weight is in no update: it stays, the others move
        assert [int((~p.isfinite()).sum()) for p in results[0]] == [1, 0, 1]


def test_lists_that_take_the_elementwise_way():
    base = torch.ones(8, 6, device=DEV)
    ok = [torch.ones(8, 6, device=DEV)]
    assert kernels.lamb_takes(ok, ok, ok, ok)
    assert not kernels.lamb_takes([base.t()], [base.t()], [base.t()], [base.t()])
    assert not kernels.lamb_takes(ok, [base.t().contiguous()], ok, ok)
    assert not kernels.lamb_takes([base.half()], ok, ok, ok)
    assert not kernels.lamb_takes([base.cpu()], [base.cpu()], [base.cpu()], [base.cpu()])
    p = torch.nn.Parameter(torch.randn(6, 8, device=DEV).t())
    q = torch.nn.Parameter(p.detach().clone(memory_format=torch.contiguous_format))
    p.grad = torch.full((8, 6), 0.5, device=DEV)
    q.grad = p.grad.clone()
    Lamb([p], lr=0.1).step()
    Lamb([q], lr=0.1).step()
    assert torch.allclose(p, q, rtol=1e-5, atol=1e-6)
