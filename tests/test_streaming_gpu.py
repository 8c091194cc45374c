"""GPU parity of the 16-bit streaming kernels: calls with more 32-token blocks than
the split kernels take, in every form that the launchers pick by length, head dim
and strides.  Each listed case names the kernels it is there for (the launched
kernels' own names, read from a trace of the call), so that a moved threshold shows
as a failure here and not as a case that tests something else.

The last test sends the random shapes of test_random_sweep_gpu, which by themselves
are small enough for the split kernels, through the same forms as one head of many.
"""
import math
import re

import numpy as np
import pytest
import torch

import rbf_attention_amd as ra
from test_parity_gpu import MODEL_RATIO, compare_case, np64, oracle_all, rand_inputs
from test_random_sweep_gpu import CASES as RANDOM_CASES

pytestmark = pytest.mark.gpu

BF, FP = torch.bfloat16, torch.float16


def launched(fn):
    """{"fwd": (features, waves, LDS-DMA buffers), "dq": the same, "dkdv": ("one" or
    "pair" waves per key block, features, buffers)} of the streaming kernels that fn
    launches; any other kernel of the library under its own name."""
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    got = {}
    for name in (e.name for e in p.events()):
        m = re.search(r"(rbf_\w+?_kernel)(?:I(?:DF16b|DF16_)((?:L[ib]\d+E)+)|<[^,>]+,([^>]*)>)", name)
        if not m:
            continue
        base = m.group(1)
        args = m.group(2) or m.group(3).replace("true", "1").replace("false", "0")
        a = [int(x) for x in re.findall(r"\d+", args)]
        if base == "rbf_fwd_kernel":
            got["fwd"] = (a[0], a[1], a[-1])
        elif base == "rbf_bwd_dq_kernel":
            got["dq"] = (a[0], a[1], a[-1])
        elif base == "rbf_bwd_dkdv_kernel":
            got["dkdv"] = ("one", a[0], a[-1])
        elif base == "rbf_bwd_dkdv_pair_kernel":
            got["dkdv"] = ("pair", a[0], a[-1])
        else:
            got[base] = a
    return got


def make(B, H, N, D, dtype, dev, layout, std, seed, key_scale):
    """q, k, v, dO as plain tensors, or as the model's views (rows of a packed
    projection; dO of a token-major output), or with q and k as a window that slides
    by eight elements per token (rows that overlap: register staging)."""
    q, k, v, do = rand_inputs(B, H, N, D, dtype, dev, std=std, seed=seed, key_scale=key_scale)
    if layout == "views":
        q, k, v = torch.stack([t.transpose(1, 2) for t in (q, k, v)], 2).permute(2, 0, 3, 1, 4)
        do = do.transpose(1, 2).contiguous().transpose(1, 2)
        assert q.stride(2) == 3 * H * D and do.stride(2) == H * D
    elif layout == "sliding":
        q, k = (torch.nn.functional.pad(t.reshape(B, H, N * D)[..., : 8 * N], (0, D)).unfold(-1, D, 8)[:, :, :N] for t in (q, k))
        assert k.stride(2) == 8
    return q, k, v, do


def run(q, k, v, do, softmax, causal, gamma, npre):
    x = [t.detach().requires_grad_() for t in (q, k, v)]
    fn = ra.run_triton_rbf if softmax else ra.run_triton_non_softmax_rbf
    out = fn(*x, causal, sm_scale=gamma, num_prefix=npre)
    return (out.detach(), *torch.autograd.grad(out, x, do))


# (B, H, N, D, dtype, softmax, causal, prefix, layout), then fwd, dq and dkdv as launched() names them
CASES = [
    # 64 features: two and three buffers, dK/dV staged through registers, by 4-wave DMA, by 8-wave DMA
    ((24, 8, 700, 64, FP, True, True, 0, "views"), (64, 4, 2), (64, 4, 3), ("one", 64, 0)),
    ((24, 8, 700, 64, BF, True, True, 300, "plain"), (64, 4, 2), (64, 4, 3), ("one", 64, 0)),
    ((24, 8, 650, 64, BF, False, False, 0, "plain"), (64, 4, 2), (64, 4, 3), ("one", 64, 0)),
    ((10, 16, 1501, 64, BF, True, False, 0, "plain"), (64, 8, 3), (64, 4, 3), ("one", 64, 2)),
    ((10, 16, 1501, 64, FP, True, True, 0, "views"), (64, 8, 3), (64, 4, 3), ("one", 64, 2)),
    ((10, 16, 1450, 64, BF, False, True, 90, "views"), (64, 4, 2), (64, 4, 3), ("one", 64, 2)),
    ((4, 16, 4100, 64, BF, True, True, 300, "views"), (64, 8, 3), (64, 4, 3), ("one", 64, 3)),
    # padded to 32 and 64 features
    ((9, 16, 901, 24, BF, True, True, 40, "views"), (32, 4, 2), (32, 4, 3), ("one", 32, 0)),
    ((12, 16, 450, 40, BF, True, True, 0, "views"), (64, 4, 2), (64, 4, 3), ("one", 64, 0)),
    ((9, 16, 1501, 48, FP, False, True, 0, "views"), (64, 8, 3), (64, 4, 3), ("one", 64, 2)),
    # 96 features, filled and not
    ((8, 12, 900, 96, BF, True, True, 0, "views"), (96, 4, 2), (96, 4, 2), ("pair", 96, 1)),
    ((8, 12, 1500, 88, FP, True, False, 0, "views"), (96, 8, 3), (96, 8, 3), ("pair", 96, 1)),
    ((6, 16, 1410, 72, BF, False, True, 200, "views"), (96, 8, 3), (96, 8, 3), ("pair", 96, 1)),
    # 128 features, filled and not: two buffers, dK/dV through registers and by DMA; three, binned and not
    ((8, 12, 777, 128, BF, True, True, 0, "views"), (128, 4, 2), (128, 4, 2), ("pair", 128, 0)),
    ((8, 16, 600, 104, BF, False, True, 0, "views"), (128, 4, 2), (128, 4, 2), ("pair", 128, 0)),
    ((8, 12, 850, 120, FP, True, True, 400, "plain"), (128, 4, 2), (128, 4, 2), ("pair", 128, 0)),
    ((8, 16, 1100, 128, FP, True, True, 0, "views"), (128, 4, 2), (128, 4, 2), ("pair", 128, 1)),
    ((5, 16, 1300, 112, BF, False, False, 0, "plain"), (128, 4, 2), (128, 4, 2), ("pair", 128, 1)),
    ((6, 16, 1500, 128, BF, True, True, 200, "views"), (128, 8, 3), (128, 8, 3), ("pair", 128, 1)),
    ((5, 12, 1500, 128, BF, True, False, 0, "views"), (128, 8, 2), (128, 8, 3), ("pair", 128, 1)),
    # rows that the LDS-DMA does not take
    ((24, 8, 700, 64, BF, True, True, 0, "sliding"), (64, 4, 0), (64, 4, 0), ("one", 64, 0)),
    ((8, 16, 900, 128, BF, False, True, 0, "sliding"), (128, 8, 0), (128, 4, 0), ("pair", 128, 0)),
    ((5, 16, 1300, 128, BF, True, True, 0, "sliding"), (128, 8, 0), (128, 8, 0), ("pair", 128, 0)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}N{}D{}_{}_{}_{}_p{}_{}".format(
    *c[0][:4], {BF: "bf16", FP: "fp16"}[c[0][4]], "sm" if c[0][5] else "ns", "causal" if c[0][6] else "full", *c[0][7:]))
def test_forms(cuda_device, case):
    """The oracle on the first and the last (b, h) slice."""
    (B, H, N, D, dtype, softmax, causal, npre, layout), fwd, dq, dkdv = case
    x = make(B, H, N, D, dtype, cuda_device, layout, 1.0 if softmax else 0.5, N + D, 0.5 if softmax and layout != "sliding" else 0.0)
    args = (softmax, causal, 0.5 / math.sqrt(D), npre)
    assert launched(lambda: run(*x, *args)) == {"fwd": fwd, "dq": dq, "dkdv": dkdv}
    outs = run(*x, *args)
    for b, h in ((0, 0), (B - 1, H - 1)):
        compare_case(*x, softmax=softmax, causal=causal, gamma=args[2], num_prefix=npre, sl=(slice(b, b + 1), slice(h, h + 1)),
                     tag=f"{case[0]} b{b}h{h}", outs=outs)


@pytest.mark.parametrize("shape,fwd", [((24, 8, 700, 64), (64, 4, 2)), ((10, 16, 1501, 64), (64, 8, 3)), ((8, 12, 900, 96), (96, 4, 2)),
                                       ((8, 12, 850, 128), (128, 4, 2)), ((6, 16, 1500, 128), (128, 8, 3)), ((5, 12, 1500, 112), (128, 8, 3))],
                         ids=str)
@pytest.mark.parametrize("shift", [3.9, 6.0])
def test_far_queries(cuda_device, shape, fwd, shift):
    """Rows whose sums leave the static bound: work-groups run again with an online
    max, through the same two or three buffers."""
    B, H, N, D = shape
    q, k, v, do = rand_inputs(B, H, N, D, BF, cuda_device, seed=17)
    q[:, ::2, : N // 3] += shift
    args = (True, True, 0.0625, 0)
    assert launched(lambda: run(q, k, v, do, *args))["fwd"] == fwd
    outs = run(q, k, v, do, *args)
    for b, h in ((0, 0), (B - 1, H - 2)):
        sl = (slice(b, b + 1), slice(h, h + 1))
        refs, _, model = oracle_all(q, k, v, do, *args[:2], args[2], 0, sl, with_model=True)
        norm = lambda x: float((x ** 2).sum() ** 0.5)  # noqa: E731
        for i in (0, 3):
            rel, rel_model = (norm(x - refs[i]) / norm(refs[i]) for x in (np64(outs[i][sl]), model[i]))
            assert rel <= MODEL_RATIO * rel_model + 1e-6, ("O" if i == 0 else "dV", rel, rel_model)
        # dQ and dK amplify the rounding of a few rows' O (through Delta) by |q| ~ 50, so
        # they are held to 64-bit arithmetic on the kernel's own O.  What is left are the
        # roundings of dS and of the result, 2^-9 each at most: 2^-8.5 = 2.8e-3 for dQ, and
        # twice that for dK, a difference of two sums (measured: 2.6e-3 and 3.7e-3 at most;
        # the rounding model on its own O: 2.6e-3 and 5.7e-3)
        qn, kn, vn, dn, on = (np64(t[b, h]) for t in (q, k, v, do, outs[0]))
        s = 2 * args[2] * (qn @ kn.T) - args[2] * (kn * kn).sum(-1)
        s[np.triu_indices(N, 1)] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        ds = p * (dn @ vn.T - (dn * on).sum(-1, keepdims=True))
        for name, got, ref, bound in (("dQ", outs[1], 2 * args[2] * (ds @ kn), 2.8e-3),
                                      ("dK", outs[2], 2 * args[2] * (ds.T @ qn - ds.sum(0)[:, None] * kn), 5.6e-3)):
            rel = norm(np64(got[b, h]) - ref) / norm(ref)
            assert rel <= bound, (name, rel)


@pytest.mark.parametrize("shape", [(24, 8, 700, 64), (8, 12, 900, 96), (8, 12, 777, 128), (6, 16, 1500, 128), (9, 16, 1501, 48)], ids=str)
def test_deterministic(cuda_device, shape):
    B, H, N, D = shape
    x = rand_inputs(B, H, N, D, BF, cuda_device, seed=21)
    a, b = (run(*x, True, True, 0.5 / math.sqrt(D), 0) for _ in range(2))
    assert all(torch.equal(s, t) for s, t in zip(a, b))


def heads_for_streaming(N, D):
    """Heads that take a call of this length and head dim past the split kernels
    (None: none do, the head-resident kernels follow them)."""
    nblk = -(-N // 32)
    width = 32 if D <= 32 else 64 if D <= 64 else 128
    need = {32: 3072, 64: 2304 if nblk >= 64 else 1408, 128: 2048}[width] // nblk + 1
    return need if N > 576 or width != 64 or need < 256 else None


@pytest.mark.parametrize("case", [c for c in RANDOM_CASES if c[5] != torch.float32 and heads_for_streaming(c[3], c[4])],
                         ids=lambda c: f"{c[0]}_N{c[3]}D{c[4]}")
def test_random_shapes_as_one_head_of_many(cuda_device, case):
    i, _, _, N, D, dtype, softmax, causal, npre, gamma, token_major = case
    q, k, v, do = rand_inputs(1, 1, N, D, dtype, cuda_device, std=1.0 if softmax else 0.5, seed=i)
    many = heads_for_streaming(N, D)
    x = [t.expand(many, 1, N, D) for t in (q, k, v, do)]
    if token_major:
        x = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in x]
    out = run(*x, softmax, causal, gamma, npre)
    assert all(torch.equal(t, t[:1].expand_as(t)) for t in out)  # every head the same
    refs, _, model = oracle_all(q, k, v, do, softmax, causal, gamma, npre, with_model=True)
    for name, got, ref, m in zip(("O", "dQ", "dK", "dV"), out, refs, model):
        norm = float((ref ** 2).sum() ** 0.5)
        if norm == 0.0 or abs(ref).max() < 1e-5:
            assert float(got[:1].abs().max()) <= 1e-4, name
            continue
        rel, rel_model = (float(((t - ref) ** 2).sum() ** 0.5) / norm for t in (np64(got[:1]), m))
        bound = 3e-2 if N <= 2 and name in ("dQ", "dK") else 1e-2
        assert rel <= max(bound, MODEL_RATIO * rel_model), (name, rel, rel_model)
        if ref.size >= 4096:
            assert rel <= 1.25 * rel_model + 1e-6, (name, rel, rel_model)
