"""The fp32 kernels' arithmetic (three bf16 parts per operand, six part products),
emulated in numpy: the parts and the bound of what the six leave out, and that the
GPU tests' bounds (tests/test_f32_gpu.py) notice the loss of any one of them."""
import math

import numpy as np
import pytest

from rbf_attention_amd import workloads as wl
from test_f32_gpu import REL

PRODUCTS = ("lh", "hl", "mm", "mh", "hm", "hh")  # (part of A, part of B), as csrc/rbf_attn_f32_kernels.h mma3


def bf16(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def cut(x):
    x = np.asarray(x, np.float32)
    h = bf16(x)
    m = bf16(x - h)
    low = (x - h) - m
    lifted = np.abs(x) >= 2.0 ** -102  # the kernels' operands are, where it counts (kLift)
    assert np.array_equal(bf16(low)[lifted], low[lifted])
    return {"h": h.astype(np.float64), "m": m.astype(np.float64), "l": low.astype(np.float64)}


def product(a, b, which):
    pa, pb = cut(a), cut(b)
    return sum(pa[t[0]] @ pb[t[1]] for t in which)


def exact_product(a, b, which):
    return np.asarray(a, np.float64) @ np.asarray(b, np.float64)


def attention(q, k, v, do, gamma, softmax, causal, npre, mul, which=None):
    """O, dQ, dK, dV of one head in 64 bits, with mul for every product."""
    i = np.arange(q.shape[0])
    vis = (i[None, :] <= i[:, None]) | (i[None, :] < npre) | (not causal)
    s = mul(q, k.T, which) - 0.5 * (k.astype(np.float64) ** 2).sum(-1)
    if softmax:
        e = np.where(vis, 2 * gamma * s, -np.inf)
        e = np.exp(e - e.max(-1, keepdims=True))
        p = e / e.sum(-1, keepdims=True)
    else:
        p = np.where(vis, np.exp(2 * gamma * (s - 0.5 * (q.astype(np.float64) ** 2).sum(-1, keepdims=True))), 0.0)
    o = mul(p, v, which)
    ds = p * (mul(do, v.T, which) - (do * o).sum(-1, keepdims=True) * softmax)
    dq = 2 * gamma * (mul(ds, k, which) - (0.0 if softmax else ds.sum(-1, keepdims=True) * q))
    dk = 2 * gamma * (mul(ds.T, q, which) - ds.sum(0)[:, None] * k)
    return o, dq, dk, mul(p.T, do, which)


def test_parts():
    """They add up exactly, and the left-out products stay below 2^-24 of the whole
    (over 2^16 mantissas, against the worst of them)."""
    bits = np.arange(0, 1 << 23, 1 << 7, dtype=np.uint32) | 0x3F800000 | 0x55
    x = bits.view(np.float32)
    p = cut(x)
    assert np.array_equal(p["h"] + p["m"] + p["l"], x.astype(np.float64))
    worst = np.argmax(np.abs(p["m"]) + 2.0 ** 9 * np.abs(p["l"]))
    for j in (worst, int(np.argmax(np.abs(p["l"]))), 0, x.size - 1):
        got = sum(p[t[0]] * p[t[1]][j] for t in PRODUCTS)
        rel = np.abs(got - x.astype(np.float64) * x[j]) / (x.astype(np.float64) * x[j])
        assert rel.max() <= 2.0 ** -24, rel.max()


@pytest.mark.parametrize("N,D,softmax,causal,npre", [(129, 64, True, False, 0), (300, 64, True, True, 70), (200, 8, True, True, 0),
                                                     (257, 40, False, True, 0), (130, 72, True, True, 0), (65, 128, False, True, 20)])
def test_every_product_counts(N, D, softmax, causal, npre):
    """With all six, the products' own error is far below the bounds; without any one
    of them every output is past its bound."""
    w = wl.Workload("adhoc", B=1, H=1, content=N, D=D, dtype="fp32", registers=0, std=1.0 if softmax else 0.5,
                    key_lognormal=0.5 if softmax else 0.0, seed=N + D)
    x = [t[0, 0].numpy() for t in wl.make_inputs(w)]
    args = (0.5 / math.sqrt(D), softmax, causal, npre)
    want = attention(*x, *args, exact_product)
    for left_out in (None, *PRODUCTS):
        got = attention(*x, *args, product, [t for t in PRODUCTS if t != left_out])
        for name, a, b in zip(("O", "dQ", "dK", "dV"), got, want):
            rel = np.linalg.norm(a - b) / np.linalg.norm(b)
            if left_out is None:
                assert rel <= 0.05 * REL[name], (name, rel)
            else:
                assert rel > REL[name], (left_out, name, rel)
