"""Softmax states at the ends of their range: every form of the attention
kernels on scores far below 0 and on a first half whose 2^score is 0 in FP32
while the second's is not.

Queries are one constant and every key block one score level, so that a block
equals its centroid and 64-bit dense attention is the result of every form at
every beta.
"""

import math

import pytest
import torch

from sol_attn_amd import _native, dense_attention, sol_attention
from sol_testlib import HAS_GPU

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not HAS_GPU, reason="AMD ROCm GPU required")]

QUERY = 4.0


def _keys(levels, tk, d, heads):
    """K [1, tk, heads, d] whose scores (log2 units, default scale) are about
    `levels` [tk], and the scores it has after the rounding to BF16."""
    k = (torch.as_tensor(levels, dtype=torch.float64) / (QUERY * d ** 0.5 * math.log2(math.e))).to(torch.bfloat16)
    return k.view(1, tk, 1, 1).expand(1, tk, heads, d).contiguous().cuda(), k.double() * QUERY * d ** 0.5


def _case(levels, tq, d, heads, seed=1):
    tk = len(levels)
    k, logits = _keys(levels, tk, d, heads)
    q = torch.full((1, tq, heads, d), QUERY, dtype=torch.bfloat16, device="cuda")
    v = torch.randn((1, tk, heads, d), generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16)
    p = torch.softmax(logits, 0)
    want = torch.einsum("t,bthd->bhd", p, v.double())[:, None].expand(1, tq, heads, d)
    return q, k, v.cuda(), want


def _close(got, want, what):
    got = got.double().cpu()
    finite = bool(torch.isfinite(got).all())
    assert finite, f"{what}: not finite"
    # BF16 probabilities and outputs, rounded by at most 2^-8 each and 2^-9 on average, and FP32 sums far below.
    rel = ((got - want).norm() / want.norm()).item()
    assert rel < 2 ** -8, f"{what}: relative error {rel:.4f}"


def _form(monkeypatch, form, q, k, v, beta, local=0, **kw):
    with monkeypatch.context() as mp:
        mp.setattr(_native, "WORKGROUP_FORM", form)
        mp.setattr(_native, "ROUTE_PREPASS", False)
        return _native.launch_sol(q, k, v, q.shape[-1] ** -0.5, beta, local, 0, kw.pop("q_sink", 0), False, **kw)[0]


def _all_forms(monkeypatch, levels, d, tq=70, heads=2, block_levels=True):
    """Every form against 64 bits.  Without `block_levels` a block's keys differ and only exact forms apply."""
    q, k, v, want = _case(levels, tq, d, heads)
    _close(dense_attention(q, k, v), want, "dense")
    for form in (1, 2):
        _close(_form(monkeypatch, form, q, k, v, -math.inf), want, f"form {form} beta -inf")
        for beta in (1.0, math.inf):
            for local in (0, 1 << 30):  # centroids but for the diagonal block; every block exact
                if block_levels or local:
                    _close(_form(monkeypatch, form, q, k, v, beta, local), want, f"form {form} beta {beta} local {local}")
    for beta in (1.0, math.inf):
        for local in (0, 1 << 30):
            if block_levels or local:
                _close(sol_attention(q, k, v, beta=beta, local_blocks=local), want, f"default beta {beta} local {local}")
    if block_levels:  # one level per block is exact in INT8 (two levels of a block are rounded to 1/127 of the larger)
        _close(_form(monkeypatch, 0, q, k, v, -math.inf, qk_precision="int8"), want, "int8")


SIZES = [(64, 64), (65, 64), (100, 64), (1024, 64), (1000, 64), (2304, 64), (9000, 64),
         (64, 128), (65, 128), (1000, 128), (2304, 128), (9000, 128)]


@pytest.mark.parametrize("tk,d", SIZES)
def test_scores_far_below_zero(tk, d, monkeypatch):
    # Every 2^score is 0 in FP32: the first keys have to move the max all the same.
    print(f"low scores: Tk{tk} D{d}", flush=True)
    levels = [-200.0 - 30.0 * (t // 64 % 3) for t in range(tk)]
    _all_forms(monkeypatch, levels, d)


@pytest.mark.parametrize("d", [64, 128])
def test_first_half_below_the_fp32_range(d, monkeypatch):
    # -130, then -124: the second half's 2^score is not 0, the first half's is.
    print(f"first half: D{d}", flush=True)
    levels = [-130.0 if t < 32 else -124.0 for t in range(64)] + [-130.0] * 64
    _all_forms(monkeypatch, levels, d, block_levels=False)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [3, 7, 14, 28, 56, 63])
def test_outputs_are_rounded_quotients(n, d, monkeypatch):
    # n equal keys whose values sum to n times a tie between two BF16 numbers: FP32 holds the sum and the quotient,
    # so the output is the tie rounded to even.  (The sum times FP32's 1 / n rounds the other way for
    # some ties at every n here but 3.)
    print(f"quotients: Tk{n} D{d}", flush=True)
    ties = (257 + 2 * torch.arange(d, dtype=torch.float64) % 254) / 256.0
    total = n * ties
    v = torch.zeros((1, n, 1, d), dtype=torch.float64)
    for t in range(3):  # 9 bits times n: two or three BF16 terms
        v[0, t, 0] = total.float().to(torch.bfloat16).double()
        total = total - v[0, t, 0]
    assert not total.any()
    v = v.to(torch.bfloat16).cuda()
    k = torch.ones((1, n, 1, d), dtype=torch.bfloat16, device="cuda")
    q = torch.zeros((1, 70, 1, d), dtype=torch.bfloat16, device="cuda")
    want = ties.float().to(torch.bfloat16).expand(1, 70, 1, d)   # round to nearest, ties to even
    for got in (dense_attention(q, k, v), sol_attention(q, k, v), _form(monkeypatch, 1, q, k, v, 1.0)):
        assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tk,heads", [(100, 2), (700, 2), (2304, 2), (2304, 150)])   # four groups; two
def test_infinite_values_stay_infinite(d, tk, heads):
    # Every block exact: one infinite value per head, in the first block (which groups that have run out of tiles
    # pass through again) and in the last.
    print(f"infinite values: D{d} Tk{tk} H{heads}", flush=True)
    q, k, v = (torch.randn((1, t, heads, d), generator=torch.Generator().manual_seed(s)).to(torch.bfloat16)
               for t, s in ((100, 4), (tk, 5), (tk, 6)))
    v[0, 3, ::2, 5], v[0, tk - 20, 1::2, 7] = math.inf, -math.inf
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    for got in (dense_attention(q, k, v), sol_attention(q, k, v, local_blocks=1 << 20)):
        got = got.float().cpu()
        assert (got[0, :, ::2, 5] == math.inf).all() and (got[0, :, 1::2, 7] == -math.inf).all()
        got[0, :, ::2, 5] = got[0, :, 1::2, 7] = 0.0
        assert torch.isfinite(got).all()
