"""fp32 values that three bf16 parts cannot carry or that lie at the ends of fp32's
range: exponentials down to 2^-125 and inputs of every magnitude keep their full
precision, infinities and NaN come out where plain arithmetic puts them, and one
such value leaves the rest of a call alone.

Bounds: elementwise and relative, from a computation in 64 bits.  The inputs are
chosen so that the exponents' rounding is small where it says so: gamma = ln 2 / 2
makes c = 2 gamma log2(e) = 1 to 2^-24, so that exponents are the products of the
inputs."""
import math

import pytest
import torch

import rbf_attention_amd as ra

pytestmark = pytest.mark.gpu

LN2_2 = math.log(2.0) / 2


def ref64(q, k, v, do, gamma, softmax, causal, npre):
    """O, dQ, dK, dV in 64 bits on the host, row sums over the visible keys only
    (0 * inf does not arise for a masked pair)."""
    q, k, v, do = (t.double().cpu() for t in (q, k, v, do))
    n = q.shape[2]
    i = torch.arange(n)
    vis = ((i[None, :] <= i[:, None]) | (i[None, :] < npre)) if causal else torch.ones(n, n, dtype=torch.bool)
    dist = (q.unsqueeze(3) - k.unsqueeze(2)).square().sum(-1)
    e = -gamma * dist
    if softmax:
        p = torch.softmax(e.masked_fill(~vis, float("-inf")), -1)
    else:
        p = torch.exp(e).masked_fill(~vis, 0.0)
    times = lambda m, x, seen: torch.where(seen.unsqueeze(-1), m.unsqueeze(-1) * x.unsqueeze(2), 0.0).sum(3)  # noqa: E731
    o = times(p, v, vis)
    dp = do @ v.transpose(-1, -2)
    ds = p * (dp - (do * o).sum(-1, keepdim=True)) if softmax else p * dp
    dq = 2 * gamma * (ds @ k - ds.sum(-1, keepdim=True) * q)
    dk = 2 * gamma * (ds.transpose(-1, -2) @ q - ds.sum(-2).unsqueeze(-1) * k)
    return o, dq, dk, times(p.transpose(-1, -2), do, vis.t())


def run(q, k, v, do, gamma, softmax=True, causal=True, npre=0):
    x = [t.clone().requires_grad_() for t in (q, k, v)]
    fn = ra.run_triton_rbf if softmax else ra.run_triton_non_softmax_rbf
    out = fn(*x, causal, sm_scale=gamma, num_prefix=npre)
    return (out.detach(), *torch.autograd.grad(out, x, do))


def rel(got, want):
    """Largest elementwise relative error."""
    want = want.double()
    err = (got.double().cpu() - want).abs()
    return float((err / want.abs()).nan_to_num(posinf=0.0).masked_fill(want == 0, 0.0).max())


def randn(gen, *shape):
    return torch.randn(shape, generator=gen)


# (B, H, N, D): four, two and one wave per block at 64 features, the other widths
SHAPES = [(1, 2, 70, 64), (4, 12, 500, 64), (7, 16, 900, 64), (2, 3, 100, 24), (3, 2, 40, 128), (6, 16, 300, 128)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("x", [100.125, 112.5, 120.125, 124.5])
def test_small_exponentials(cuda_device, shape, x):
    """Non-softmax: every key at the same distance, P = 2^-x; the outputs are P times
    plain sums.  Softmax: keys that no query attends to, P = 2^-x, have a dV of P
    times a plain sum.  v and dO are positive, so that the sums do not cancel.  The
    hardware's exponential is good to 1 ulp, the sums to ~2^-22."""
    B, H, N, D = shape
    g = torch.Generator().manual_seed(1)
    v, do = (torch.rand(B, H, N, D, generator=g) + 0.5 for _ in range(2))
    q = torch.zeros(B, H, N, D)
    k = torch.zeros(B, H, N, D)
    q[..., 0] = math.sqrt(2 * x)  # c * 0.5 * ||q||^2 = x
    dev = [t.to(cuda_device) for t in (q, k, v, do)]
    sl = (slice(B - 1, B), slice(H - 1, H))
    want = ref64(*(t[sl] for t in (q, k, v, do)), LN2_2, False, True, 0)
    got = run(*dev, LN2_2, softmax=False)
    # sqrt(2x) rounded to fp32 moves x by 2^-24 relative: x * 2^-24 * 2 * ln 2 of P
    tol = 2e-5
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, want):
        assert rel(a[sl], b) <= tol, (name, rel(a[sl], b))
    # softmax: the queries sit on key 0; the others are x away
    q.zero_()
    k[:, :, 1:, 0] = math.sqrt(2 * x)
    dev = [t.to(cuda_device) for t in (q, k, v, do)]
    want = ref64(*(t[sl] for t in (q, k, v, do)), LN2_2, True, True, 0)
    got = run(*dev, LN2_2)
    assert rel(got[3][sl], want[3]) <= tol, rel(got[3][sl], want[3])
    # dK of such a key is 2 gamma (0 - sum(dS) k): relative to its largest entries
    a, b = got[2][sl].double().cpu()[..., 1:, 0], want[2][..., 1:, 0]
    assert float((a - b).norm() / b.norm()) <= 1e-4


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("which,scale", [("v", 2.0 ** -118), ("v", 2.0 ** 60), ("do", 2.0 ** -118), ("do", 2.0 ** 60), ("v", 2.0 ** 21)])
def test_magnitudes(cuda_device, shape, softmax, which, scale):
    """v or dO scaled by a power of two scales what is linear in it, to the last bits
    (the smallest outputs fall below fp32's normal range: an absolute floor)."""
    B, H, N, D = shape
    g = torch.Generator().manual_seed(2)
    q, k, v, do = (randn(g, B, H, N, D).to(cuda_device) * 0.5 for _ in range(4))
    gamma = 0.5 / math.sqrt(D)
    base = run(q, k, v, do, gamma, softmax)
    if which == "v":
        got = run(q, k, v * scale, do, gamma, softmax)
        scaled = [True, True, True, False]
    else:
        got = run(q, k, v, do * scale, gamma, softmax)
        scaled = [False, True, True, True]
    for name, a, b, s in zip(("O", "dQ", "dK", "dV"), got, base, scaled):
        want = b.double() * (scale if s else 1.0)
        err = float((a.double() - want).norm() / want.norm())
        assert err <= 4e-6, (name, err)


@pytest.mark.parametrize("shape", SHAPES[:2] + SHAPES[3:5], ids=str)
@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_non_finite(cuda_device, shape, softmax, value):
    """One non-finite element of v, or of dO: the outputs it reaches are what 64-bit
    arithmetic gives, the others those of a call without it."""
    B, H, N, D = shape
    g = torch.Generator().manual_seed(3)
    q, k, v, do = (randn(g, B, H, N, D) * 0.3 for _ in range(4))
    gamma, j, d = 0.5 / math.sqrt(D), N // 3, D // 2
    sl = (slice(B - 1, B), slice(H - 1, H))
    for which in ("v", "do"):
        t = {"v": v.clone(), "do": do.clone()}
        t[which][B - 1, H - 1, j, d] = value
        got = run(*(x.to(cuda_device) for x in (q, k, t["v"], t["do"])), gamma, softmax)
        base = run(*(x.to(cuda_device) for x in (q, k, v, do)), gamma, softmax)
        want = ref64(q[sl], k[sl], t["v"][sl], t["do"][sl], gamma, softmax, True, 0)
        for name, a, b, w in zip(("O", "dQ", "dK", "dV"), got, base, want):
            # every other (b, h) is untouched
            rest = torch.ones(B, H, dtype=torch.bool)
            rest[B - 1, H - 1] = False
            assert torch.equal(a[rest.to(cuda_device)], b[rest.to(cuda_device)]), (which, name)
            if name in ("dQ", "dK") or math.isnan(value):
                continue  # sums over NaN and infinities of both signs
            a = a[sl].double().cpu()
            fin = torch.isfinite(w)
            assert torch.equal(torch.isfinite(a), fin), (which, name)
            assert torch.equal(a[~fin], w[~fin]), (which, name)
            assert float((a[fin] - w[fin]).norm() / w[fin].norm()) <= 4e-6, (which, name)


def test_one_value_leaves_the_rest_alone(cuda_device):
    """A tiny and a huge element among ordinary ones: within the ordinary bound."""
    B, H, N, D = 2, 3, 200, 64
    g = torch.Generator().manual_seed(4)
    q, k, v, do = (randn(g, B, H, N, D) for _ in range(4))
    v[0, 0, 5, 3] = 2.0 ** -120
    do[1, 2, 150, 7] = 2.0 ** -125
    v[1, 0, 77, 1] = 3e9
    gamma = 0.0625
    got = run(*(x.to(cuda_device) for x in (q, k, v, do)), gamma)
    want = ref64(q, k, v, do, gamma, True, True, 0)
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, want):
        for h in range(H):
            for i in range(B):
                x, y = a[i, h].double().cpu(), b[i, h]
                assert float((x - y).norm() / y.norm()) <= 1e-5, (name, i, h)
