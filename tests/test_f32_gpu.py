"""GPU parity of the fp32 kernels (three bf16 parts per operand) against the
float64 oracle, at the edges of their tiles, head-dim widths and of the block
counts at which the launchers change the split.

Bounds beside the max-abs <= 1e-4 of tests/test_parity_gpu.py, on the relative
2-norm (REL).  An exponential's argument is an fp32 sum of terms up to ~2^6 in base
2 here, so it carries up to ~2^-18 = 4e-6 of rounding (typically a quarter of it),
which is the relative error of P; dS adds the rounding of dP - Delta, whose terms
cancel by a few times, and the products' own sums add 2^-24 per term.  Measured on
these cases: O up to 0.81e-6, dQ 1.92e-6, dK 2.0e-6, dV 1.85e-6, as with plain fp32
matrix instructions.  The bounds lie just above, below what the loss of any one
of the kernels' six part products gives (tests/test_f32_parts_cpu.py: from 1.9e-6,
2.6e-6, 3.0e-6 and 2.2e-6 on, each beside the rounding above).
"""
import math

import pytest
import torch

from test_parity_gpu import compare_case, np64, oracle_all, rand_inputs

pytestmark = pytest.mark.gpu

REL = {"O": 1.5e-6, "dQ": 2.5e-6, "dK": 2.5e-6, "dV": 2.25e-6}

# (B, H, N, D, softmax, causal, num_prefix)
CASES = [
    (1, 1, 1, 64, True, True, 0),
    (2, 3, 31, 64, True, True, 0),
    (2, 3, 33, 64, False, True, 0),
    (1, 2, 129, 64, True, False, 0),
    (1, 2, 300, 64, True, True, 70),
    (4, 10, 513, 64, True, True, 0),  # 680 blocks: past the four-way split
    (4, 10, 513, 64, False, False, 0),
    (5, 8, 1030, 64, True, True, 0),  # 1320
    (7, 16, 900, 64, True, True, 0),  # 3248: one wave per block
    (7, 16, 900, 64, False, True, 3),
    (1, 4, 200, 8, True, True, 0),
    (3, 9, 800, 24, True, True, 0),
    (1, 2, 257, 40, False, True, 0),
    (1, 2, 130, 72, True, True, 0),
    (2, 2, 65, 128, False, True, 20),
    (3, 16, 450, 128, True, True, 0),  # 720: one wave per block at 128 features
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}N{}D{}_{}_{}_p{}".format(
    *c[:4], "sm" if c[4] else "ns", "causal" if c[5] else "full", c[6]))
def test_fp32(cuda_device, case):
    """The oracle on the first, the last and one middle (b, h) slice."""
    B, H, N, D, softmax, causal, npre = case
    q, k, v, do = rand_inputs(B, H, N, D, torch.float32, cuda_device, std=1.0 if softmax else 0.5, seed=N + D,
                              key_scale=0.5 if softmax else 0.0)
    gamma, outs = 0.5 / math.sqrt(D), None
    for b, h in sorted({(0, 0), (B // 2, H // 2), (B - 1, H - 1)}):
        sl = (slice(b, b + 1), slice(h, h + 1))
        outs = compare_case(q, k, v, do, softmax=softmax, causal=causal, gamma=gamma, num_prefix=npre, sl=sl,
                            tag=f"{case} b{b}h{h}", outs=outs)
        if N > 2:
            refs, _, _ = oracle_all(q, k, v, do, softmax, causal, gamma, npre, sl, with_model=True)
            for name, got, ref in zip(("O", "dQ", "dK", "dV"), outs, refs):
                d = np64(got[sl]) - ref
                rel = float((d ** 2).sum() ** 0.5 / max((ref ** 2).sum() ** 0.5, 1e-30))
                assert rel <= REL[name], (name, rel)


@pytest.mark.parametrize("shift", [3.9, 6.0])
def test_fp32_far_queries_at_every_split(cuda_device, shift):
    """Row sums that leave the static bound make a work-group run again with a
    running max, whose partials are merged by their own offsets."""
    for B, H, N in ((1, 2, 200), (6, 12, 300), (10, 40, 260)):
        q, k, v, do = rand_inputs(B, H, N, 64, torch.float32, cuda_device, seed=17)
        q[:, ::2, :90] += shift
        for b, h in ((0, 0), (B - 1, H - 2)):
            compare_case(q, k, v, do, gamma=0.0625, sl=(slice(b, b + 1), slice(h, h + 1)), tag=f"far{shift} {B}x{H}x{N}",
                         ill_conditioned=True)
