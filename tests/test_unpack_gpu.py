"""The packed gradient of q, k and v (ops.unpack_qkv) against plain views of the
same projection output, bit for bit: the attention's own gradients, with one of
the three used elsewhere too (its gradient is then a sum), with one unused, and
with gradients asked for at the views.  A gradient that a program gets hold of
shares its memory with no other."""
import pytest
import torch

import rbf_attention_amd as ra
from rbf_attention_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("B,N,H,D,pos", [(2, 70, 3, 64, False), (1, 33, 2, 64, True), (2, 40, 2, 20, False),
                                         (32, 130, 8, 64, True), (1, 1, 1, 64, False)])
@pytest.mark.parametrize("use", ["plain", "v_twice", "q_only"])
def test_packed_gradient(cuda_device, softmax, B, N, H, D, pos, use):
    g = torch.Generator().manual_seed(N)
    qkv = (torch.randn(B, N, 3, H, D, generator=g) * 0.5).to(torch.bfloat16).to(cuda_device)
    do = torch.randn(B, H, N, D, generator=g).to(torch.bfloat16).to(cuda_device)
    P = torch.randn(1, H, N, D, generator=g).to(torch.bfloat16).to(cuda_device) if pos else None
    fn = ra.run_triton_rbf if softmax else ra.run_triton_non_softmax_rbf
    got = []
    for split in (ops.unpack_qkv, lambda t: t.permute(2, 0, 3, 1, 4).unbind(0)):
        x = qkv.clone().requires_grad_(True)
        p = P.clone().requires_grad_(True) if pos else None
        q, k, v = split(x * 1.0)
        assert q.shape == (B, H, N, D) and q.stride() == (N * 3 * H * D, D, 3 * H * D, 1)
        if use == "q_only":
            k, v = k.detach(), v.detach()
        else:
            q.retain_grad()
            v.retain_grad()
        out = fn(q, k, v, True, pos=p)
        if use == "v_twice":
            out = out + v * 0.5
        out.backward(do)
        got.append([out.detach(), x.grad] + ([p.grad] if pos else []) + ([] if use == "q_only" else [q.grad, v.grad]))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_packed_gradient_with_a_graph(cuda_device):
    """create_graph: the views' own path stays differentiable."""
    got = []
    for split in (ops.unpack_qkv, lambda t: t.permute(2, 0, 3, 1, 4).unbind(0)):
        x = torch.linspace(-1, 1, 2 * 5 * 3 * 2 * 8, device=cuda_device).view(2, 5, 3, 2, 8).requires_grad_(True)
        q, k, v = split(x * 1.0)
        (g,) = torch.autograd.grad((q * v * v).sum(), x, create_graph=True)
        (h,) = torch.autograd.grad((g * g).sum(), x)
        got.append((g.detach(), h))
    assert all(torch.equal(a, b) for a, b in zip(*got))


def inputs(dev, B=2, N=40, H=2, D=64):
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(B, N, 3, H, D, generator=g).to(dev, torch.bfloat16)
    return qkv, torch.randn(B, H, N, D, generator=g).to(dev, torch.bfloat16)


def shares(a, b):
    return a.untyped_storage().data_ptr() == b.untyped_storage().data_ptr()


def test_gradient_kept_by_a_hook(cuda_device):
    """A leaf's gradient is added to in place by the next backward pass; what a
    hook kept of the first pass stays what it was."""
    qkv, do = inputs(cuda_device)
    x = qkv.clone().requires_grad_(True)
    for keep in (lambda g: g, lambda g: g[0], lambda g: g.detach()):
        kept = []
        x.grad = None
        for _ in range(2):
            q, k, v = ops.unpack_qkv(x)
            if not kept:
                q.register_hook(lambda g: kept.append((keep(g), g.clone())))
            ra.run_triton_rbf(q, k, v).backward(do)
        view, copy = kept[0]
        assert torch.equal(view, copy if view.dim() == 4 else copy[0])
        assert not shares(view, x.grad)


@pytest.mark.parametrize("at", ["tensor", "node", "attention_node"])
def test_gradient_kept_by_node_hooks(cuda_device, at):
    qkv, do = inputs(cuda_device)
    x = qkv.clone().requires_grad_(True)
    q, k, v = ops.unpack_qkv(x)
    out = ra.run_triton_rbf(q, k, v)
    kept = []
    if at == "tensor":
        q.retain_grad()
        v.register_hook(kept.append)
    elif at == "node":
        q.grad_fn.register_prehook(lambda grads: kept.extend(grads))
    else:
        out.grad_fn.register_hook(lambda grad_inputs, _: kept.extend(grad_inputs[:3]))
    out.backward(do)
    assert kept and not any(shares(g, x.grad) for g in kept)
    if at == "tensor":
        assert not shares(q.grad, x.grad)
        # and a kept dv holds its own memory only
        assert kept[0].untyped_storage().nbytes() == kept[0].numel() * kept[0].element_size()


@pytest.mark.parametrize("ask", ["q", "q_x", "x_q_k_v"])
def test_gradients_asked_for_together(cuda_device, ask):
    """autograd.grad at the views and at the packed tensor: writing to one result
    leaves the others alone, each holds its own memory, and the values are those
    of plain views."""
    qkv, do = inputs(cuda_device)
    results = []
    for split in (ops.unpack_qkv, lambda t: t.permute(2, 0, 3, 1, 4).unbind(0)):
        x = qkv.clone().requires_grad_(True)
        q, k, v = split(x)
        wrt = {"q": (q,), "q_x": (q, x), "x_q_k_v": (x, q, k, v)}[ask]
        results.append(torch.autograd.grad(ra.run_triton_rbf(q, k, v), wrt, do))
    ours, plain = results
    assert all(torch.equal(a, b) for a, b in zip(ours, plain))
    for i, g in enumerate(ours):
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()
        others = [o.clone() for j, o in enumerate(ours) if j != i]
        g.zero_()
        assert all(torch.equal(o, c) for o, c in zip((o for j, o in enumerate(ours) if j != i), others))


def test_packed_gradient_is_not_copied(cuda_device):
    """Nothing else asks for dq, dk and dv: one buffer is written, no other of its
    size is allocated."""
    qkv, do = inputs(cuda_device, 8, 256, 8, 64)
    x = qkv.clone().requires_grad_(True)
    peaks = []
    for split in (ops.unpack_qkv, lambda t: t.permute(2, 0, 3, 1, 4).unbind(0)):
        for _ in range(2):  # the first pass loads kernels
            x.grad = None
            out = ra.run_triton_rbf(*split(x))
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            base = torch.cuda.memory_allocated()
            out.backward(do)
            peak = torch.cuda.max_memory_allocated() - base
        peaks.append(peak / x.nbytes)
    assert peaks[0] < 1.2 and peaks[1] > 1.9, peaks


def test_forward_mode_and_batched_gradients(cuda_device):
    """As plain views: tangents of a dual tensor, and a batch of gradients."""
    import torch.autograd.forward_ad as fwad

    g = torch.Generator().manual_seed(3)
    x, t = (torch.randn(2, 5, 3, 2, 8, generator=g).to(cuda_device) for _ in range(2))
    cot = torch.randn(4, 2, 2, 5, 8, generator=g).to(cuda_device)
    results = []
    for split in (ops.unpack_qkv, lambda t: t.permute(2, 0, 3, 1, 4).unbind(0)):
        with fwad.dual_level():
            q, k, v = split(fwad.make_dual(x, t))
            tangent = fwad.unpack_dual(q * k + v).tangent
        leaf = x.clone().requires_grad_(True)
        q, k, v = split(leaf)
        (batch,) = torch.autograd.grad(q * k + v, leaf, cot, is_grads_batched=True)
        results.append((tangent, batch))
    assert all(torch.equal(a, b) for a, b in zip(*results))
