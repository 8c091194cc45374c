"""torch.jit.trace of the public calls on the GPU: values and gradients of the
traced function equal the eager ones (same kernels, so bit for bit)."""
import pytest
import torch

import rbf_attention_amd as ra
from rbf_attention_amd.model import RBFAttention

pytestmark = pytest.mark.gpu


def randn(dev, seed, *shape, dtype=torch.bfloat16, grad=True):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(dev, dtype).requires_grad_(grad)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("fn,kw", [(ra.run_triton_rbf, {}), (ra.run_triton_non_softmax_rbf, {}),
                                   (ra.run_triton_rbf, {"sm_scale": 0.0625, "num_prefix": 3, "token_major": True})])
def test_attention(cuda_device, fn, kw, grad):
    call = lambda q, k, v: fn(q, k, v, True, **kw)  # noqa: E731
    new = lambda s: [randn(cuda_device, 3 * s + i, 2, 3, 70, 64, grad=grad) for i in range(3)]  # noqa: E731
    traced = torch.jit.trace(call, new(0))
    x = new(1)
    want, got = call(*x), traced(*x)
    assert torch.equal(got, want)
    if grad:
        do = randn(cuda_device, 9, 2, 3, 70, 64, grad=False)
        for a, b in zip(torch.autograd.grad(got, x, do), torch.autograd.grad(want, x, do)):
            assert torch.equal(a, b)


def test_module(cuda_device):
    torch.manual_seed(0)
    m = RBFAttention(4, 256, max_seq_len=128, num_registers=2, pos_weight_init=1.0).to(cuda_device, torch.bfloat16)
    new = lambda s: randn(cuda_device, s, 2, 60, 256)  # noqa: E731
    traced = torch.jit.trace(m, (new(1),))
    x = new(2)
    want, got = m(x), traced(x)
    assert torch.equal(got, want)
    dy = randn(cuda_device, 3, 2, 60, 256, grad=False)
    (a,), (b,) = torch.autograd.grad(got, x, dy), torch.autograd.grad(want, x, dy)
    assert torch.equal(a, b)


def test_decode(cuda_device):
    new = lambda s: [randn(cuda_device, s, 2, 3, 1, 64, grad=False)] + [  # noqa: E731
        randn(cuda_device, s + i, 2, 3, 50, 64, grad=False) for i in (1, 2)]
    traced = torch.jit.trace(lambda q, k, v: ra.rbf_decode(q, k, v), new(0))
    x = new(5)
    for a, b in zip(traced(*x), ra.rbf_decode(*x)):
        assert torch.equal(a, b)
