"""Infinities and NaN in one element of v, dO or k, in each kernel form: the outputs
they reach are those of 64-bit arithmetic (infinite with its sign, or NaN), every
other one is what it is without them.  Every key is visible, so that no masked pair
(P = 0 against an infinity) is among the products.  And the split kernels' row
terms, which are put together from three bf16 values, against the streaming
kernels' on the same head."""
import math

import pytest
import torch

import rbf_attention_amd as ra

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16

# (B, H, N, D, dtype): four and two waves per block; streaming at 64 features with two
# and three buffers, register-staged dK/dV, 96 features, 128 features short and long
FORMS = [
    (1, 2, 70, 64, BF), (1, 3, 70, 32, FP), (1, 2, 100, 128, BF), (4, 11, 513, 64, BF), (4, 8, 900, 64, FP), (2, 9, 450, 96, BF),
    (24, 8, 700, 64, BF), (7, 16, 1501, 64, FP), (8, 12, 777, 96, BF), (4, 16, 1500, 80, FP), (12, 16, 450, 128, BF), (5, 12, 1400, 128, BF),
]


def ref64(q, k, v, do, gamma, softmax):
    q, k, v, do = (t.double() for t in (q, k, v, do))
    s = 2 * gamma * (q @ k.t()) - gamma * (k * k).sum(-1) - gamma * (q * q).sum(-1, keepdim=True)
    p = torch.softmax(s, -1) if softmax else s.exp()
    o = p @ v
    return o, p.t() @ do


def run(x, gamma, softmax):
    leaves = [t.clone().requires_grad_() for t in x[:3]]
    fn = ra.run_triton_rbf if softmax else ra.run_triton_non_softmax_rbf
    out = fn(*leaves, False, sm_scale=gamma)
    return (out.detach(), *torch.autograd.grad(out, leaves, x[3]))


@pytest.mark.parametrize("form", FORMS, ids=str)
@pytest.mark.parametrize("softmax", [True, False])
def test_one_element(cuda_device, form, softmax):
    B, H, N, D, dtype = form
    g = torch.Generator(device=cuda_device).manual_seed(N)
    clean = [(torch.randn(B, H, N, D, generator=g, device=cuda_device) * 0.3).to(dtype) for _ in range(4)]
    gamma, at = 0.5 / math.sqrt(D), (B - 1, H - 1, N // 3, D // 2)
    base = run(clean, gamma, softmax)
    others = torch.ones(B, H, dtype=torch.bool, device=cuda_device)
    others[B - 1, H - 1] = False
    for which in (1, 2, 3):  # k, v, dO
        for value in (float("inf"), float("-inf"), float("nan")):
            x = [t.clone() if i == which else t for i, t in enumerate(clean)]
            x[which][at] = value
            got = run(x, gamma, softmax)
            what = ("q", "k", "v", "dO")[which], value
            for name, a, b in zip(("O", "dQ", "dK", "dV"), got, base):
                assert torch.equal(a[others], b[others]), (*what, name)
            want = ref64(*(t[B - 1, H - 1] for t in x), gamma, softmax)
            for name, a, w in (("O", got[0], want[0]), ("dV", got[3], want[1])):
                a = a[B - 1, H - 1].double()
                fin = torch.isfinite(w)
                assert torch.equal(torch.isfinite(a), fin), (*what, name)
                inf = torch.isinf(w)
                if which != 1:  # k: an infinite or NaN logit, by the order of the sums
                    assert torch.equal(a[inf], w[inf]), (*what, name)
                if fin.any():
                    assert float((a[fin] - w[fin]).norm() / w[fin].norm()) <= 1e-2, (*what, name)
            if which == 3:
                # dQ: the row of that query only; dK sees it everywhere
                a, b = got[1][B - 1, H - 1], base[1][B - 1, H - 1]
                rows = torch.arange(N, device=cuda_device) != at[2]
                assert torch.equal(a[rows], b[rows]) and not torch.isfinite(a[at[2]]).all(), what


@pytest.mark.parametrize("H,N,D,dtype", [(3, 200, 64, BF), (8, 700, 64, FP), (2, 300, 128, BF), (4, 500, 32, FP)])
def test_infinite_delta(cuda_device, H, N, D, dtype):
    """Delta = rowsum(O dO) of either sign enters dP as it is: the split kernels give
    infinities and NaN where the streaming kernel does (the same heads, with more of
    them in the call)."""
    g = torch.Generator(device=cuda_device).manual_seed(N)
    q, k, v, do = ((torch.randn(1, H, N, D, generator=g, device=cuda_device) * 0.3).to(dtype) for _ in range(4))
    gamma = 0.5 / math.sqrt(D)
    out, lse = torch.ops.rbf_attn_amd.scaled_fwd_ex(q, k, v, True, gamma, 0)
    out[0, 0, 10, 3] = float("inf")
    out[0, 1, N - 5, 1] = float("-inf")
    many = -(-6000 // (H * (N // 32)))
    small = torch.ops.rbf_attn_amd.scaled_bwd_ex(q, k, v, out, lse, do, True, gamma, 0)
    big = torch.ops.rbf_attn_amd.scaled_bwd_ex(*(t.expand(many, *t.shape[1:]) for t in (q, k, v, out, lse, do)), True, gamma, 0)
    for name, a, b in zip(("dQ", "dK", "dV"), small, big):
        a, b = a[0], b[0]
        assert torch.equal(torch.isnan(a), torch.isnan(b)), name
        inf = torch.isinf(b)
        assert torch.equal(torch.isinf(a), inf) and torch.equal(a[inf], b[inf]), name
    assert not torch.isfinite(small[0][0, 0, 10]).any() and torch.isfinite(small[2]).all()


@pytest.mark.parametrize("H,N,D,dtype", [(3, 200, 64, BF), (8, 900, 64, FP), (2, 300, 128, BF), (4, 500, 32, FP)])
def test_row_terms_are_exact(cuda_device, H, N, D, dtype):
    """dP - Delta with Delta hundreds of times the difference: both kernels take Delta
    and L to fp32.  Their sums differ in order: ~2^-23 of Delta, against a difference
    of 2^-9 of it, so ~1e-4 of dS.  A Delta cut to 16 bits would be 2^-16 / 2^-9 = 8e-3
    off, one to 8 bits useless."""
    g = torch.Generator(device=cuda_device).manual_seed(N)
    q, k, v, do = (torch.randn(1, H, N, D, generator=g, device=cuda_device) for _ in range(4))
    v = v * 0.25 + 40.0
    do = do * 0.25 + 1.0
    q, k, v, do = (t.to(dtype) for t in (q * 0.5, k * 0.5, v, do))
    gamma = 0.5 / math.sqrt(D)
    out, lse = torch.ops.rbf_attn_amd.scaled_fwd_ex(q, k, v, True, gamma, 0)
    many = -(-6000 // (H * (N // 32)))
    small = torch.ops.rbf_attn_amd.scaled_bwd_ex(q, k, v, out, lse, do, True, gamma, 0)
    big = torch.ops.rbf_attn_amd.scaled_bwd_ex(*(t.expand(many, *t.shape[1:]) for t in (q, k, v, out, lse, do)), True, gamma, 0)
    for name, a, b in zip(("dQ", "dK", "dV"), small, big):
        rel = float((a[0].double() - b[0].double()).norm() / b[0].double().norm())
        print(f"{name} {rel:.2e}")
        assert rel <= 5e-4, (name, rel)


@pytest.mark.parametrize("dtype,D", [(BF, 64), (FP, 128), (torch.float32, 64), (BF, 96), (BF, 256)])
@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("T,L", [(1, 50), (2, 128), (5, 256), (1, 700)])
def test_decode(cuda_device, dtype, D, softmax, T, L):
    """One split and several: an infinity in a visible key's v reaches that feature of
    that head; what the cache holds past a sequence's length reaches nothing."""
    g = torch.Generator(device=cuda_device).manual_seed(L)
    B, H = 3, 2
    q, k, v = ((torch.randn(B, H, n, D, generator=g, device=cuda_device) * 0.3).to(dtype) for n in (T, L, L))
    lens = torch.tensor([L, max(T, L // 2), max(T, L - 3)], device=cuda_device, dtype=torch.int32)
    kw = {"softmax": softmax, "sm_scale": 0.5 / math.sqrt(D)}
    base, lse = ra.rbf_decode(q, k, v, lens, **kw)
    assert torch.isfinite(base).all()
    for value in (float("inf"), float("nan")):
        k2, v2 = k.clone(), v.clone()
        for b in (1, 2):
            k2[b, :, int(lens[b]):] = value
            v2[b, :, int(lens[b]):] = value
        out, lse2 = ra.rbf_decode(q, k2, v2, lens, **kw)
        assert torch.equal(out, base) and (not softmax or torch.equal(lse, lse2)), value
    v2 = v.clone()
    v2[0, 1, 7, 5] = float("-inf")
    out, _ = ra.rbf_decode(q, k, v2, lens, **kw)
    hit = torch.zeros_like(out, dtype=torch.bool)
    hit[0, 1, :, 5] = True
    assert torch.equal(out[~hit], base[~hit]) and (out[hit] == float("-inf")).all()
