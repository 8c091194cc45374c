"""Saved-tensor hooks around the wrappers: the backward pass checks what the hooks
bring back before a kernel reads it, and takes any layout.  And views whose
memory holds the negated values."""
import pytest
import torch

import rbf_attention_amd as ra

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def make(dev, softmax, pos, D=64):
    g = torch.Generator().manual_seed(2)
    x = [torch.randn(2, 3, 50, D, generator=g).to(dev, BF).requires_grad_() for _ in range(3)]
    p = torch.randn(1, 3, 50, D, generator=g).to(dev, BF).requires_grad_() if pos else None
    do = torch.randn(2, 3, 50, D, generator=g).to(dev, BF)
    fn = ra.run_triton_rbf if softmax else ra.run_triton_non_softmax_rbf
    return x, p, do, lambda: fn(*x, True, pos=p)


CHANGES = {
    "dtype": (lambda t: t.to(torch.float16 if t.dtype == BF else torch.float64), TypeError),
    "shorter": (lambda t: t[:, :, :-1], ValueError),
    "flat": (lambda t: t.reshape(-1), ValueError),
    "batch": (lambda t: t[:1].clone(), ValueError),
    "host": (lambda t: t.cpu(), (ValueError, RuntimeError)),
}


@pytest.mark.parametrize("change", sorted(CHANGES))
@pytest.mark.parametrize("softmax", [True, False])
def test_changed_tensors_are_refused(cuda_device, softmax, change):
    """Each saved tensor in turn comes back changed (all but a shared position
    term, whose batch is 1 as it is)."""
    fn, error = CHANGES[change]
    for which in range(6 if softmax else 4):  # q, k, v, pos, out, L
        if change == "batch" and which == 3:
            continue
        x, p, do, call = make(cuda_device, softmax, True)
        n = iter(range(100))
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (next(n), t), lambda it: fn(it[1]) if it[0] == which else it[1]):
            out = call()
        with pytest.raises(error):
            out.backward(do)


@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("pos", [False, True])
def test_other_layouts(cuda_device, softmax, pos):
    """Tensors that come back with other strides, and saved on the host."""

    def strided(t):
        wide = t.new_full((*t.shape, 2), float("nan"))
        wide[..., 0] = t
        return wide[..., 0]

    results = []
    for hooks in (None, torch.autograd.graph.saved_tensors_hooks(lambda t: t, strided), torch.autograd.graph.save_on_cpu()):
        x, p, do, call = make(cuda_device, softmax, pos)
        if hooks is None:
            out = call()
        else:
            with hooks:
                out = call()
        out.backward(do)
        results.append([t.grad for t in x] + ([p.grad] if pos else []))
    for r in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, results[0]))


def test_negative_views(cuda_device):
    """As inputs and as the output's gradient, through the wrapper, the op and the
    autograd.Function alias."""
    x, _, do, _ = make(cuda_device, True, False)
    neg = lambda t: torch._neg_view(-t.detach())  # noqa: E731
    for fn in (ra.run_triton_rbf, lambda *a: torch.ops.rbf_attn_v5.scaled_fwd(*a, True)[0], ra.TritonRBFAttention.apply):
        results = []
        for view in (lambda t: t.detach(), neg):
            leaves = [view(t).requires_grad_() for t in x]
            out = fn(*leaves)
            results.append([out.detach(), *torch.autograd.grad(out, leaves, view(do))])
        assert all(torch.equal(a, b) for a, b in zip(*results))
    q, k, v = (t.detach() for t in x)
    for a, b in zip(ra.rbf_decode(q[:, :, :2], k, v), ra.rbf_decode(neg(q[:, :, :2]), neg(k), neg(v))):
        assert torch.equal(a, b)
