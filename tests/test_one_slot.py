"""One-block workgroups (a K and a V slot each) where their stream can go
wrong: scores that keep growing (a half's raw scores re-formed from global
memory), streams of one tile, partial last blocks, many centroid tiles, and
indexed windows whose key blocks are read from rows, from tiles or from both.

Every comparison is with another form of the same arithmetic (the dense
kernel, two-block workgroups, or windows with every block copied to tiles),
whose results are bit-identical by design.
"""

import math

import numpy as np
import pytest
import torch

from sol_attn_amd import IndexedPlan, _native, dense_attention, sol_attention_indexed
from sol_testlib import HAS_GPU, assert_close, block_smooth, tensors

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not HAS_GPU, reason="AMD ROCm GPU required")]


def _launch(q, k, v, form, monkeypatch, beta, **kw):
    with monkeypatch.context() as mp:
        mp.setattr(_native, "WORKGROUP_FORM", form)
        mp.setattr(_native, "ROUTE_PREPASS", False)
        return _native.launch_sol(q, k, v, q.shape[-1] ** -0.5, beta, kw.get("local", 1), kw.get("kv_sink", 0),
                                  kw.get("q_sink", 0), True)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tk", [64, 65, 127, 700, 4133])
def test_growing_scores_equal_dense(d, tk, monkeypatch):
    # Keys that grow along the sequence: the running max moves by far more
    # than the lazy slack again and again, in every tile's both halves.
    print(f"growing scores: D{d} Tk{tk}", flush=True)
    q, k, v = tensors(150, tk, d, 1, 2, device="cuda", seed=11)
    ramp = torch.linspace(0.0, 40.0, tk, device="cuda").view(1, tk, 1, 1)
    k = (k.float() * ramp).to(torch.bfloat16)
    got, counts = _launch(q, k, v, 1, monkeypatch, -math.inf)
    assert torch.equal(got, dense_attention(q, k, v))
    assert (counts == -(-tk // 64)).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tq,tk", [(64, 64), (200, 100), (130, 4096), (70, 4097), (333, 9000), (64, 12345)])
@pytest.mark.parametrize("beta", [0.5, math.inf])
def test_forms_agree(d, tq, tk, beta, monkeypatch):
    print(f"forms: D{d} Tq{tq} Tk{tk} beta {beta}", flush=True)
    q, k, v = (block_smooth(1, t, 3, d, seed=s, device="cuda") for t, s in ((tq, 1), (tk, 2), (tk, 3)))
    for local, kv_sink, q_sink in ((0, 0, 0), (1, 64, min(64, tq))):
        kw = dict(local=local, kv_sink=min(kv_sink, tk), q_sink=q_sink)
        one, c1 = _launch(q, k, v, 1, monkeypatch, beta, **kw)
        two, c2 = _launch(q, k, v, 2, monkeypatch, beta, **kw)
        assert torch.equal(c1, c2)
        assert torch.equal(one, two)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tq,tk,heads", [
    (130, 130, 2), (1100, 1090, 3), (700, 2304, 1),  # one centroid tile: three early blocks, partial last blocks
    (64, 4097, 2), (400, 8192, 3), (300, 8200, 1),   # two and three
    (200, 12288, 2), (200, 12289, 2),                # three and four (none early)
    (4160, 1100, 6),                                 # two groups
])
def test_early_local_blocks_of_small_launches(d, tq, tk, heads, monkeypatch):
    # Local blocks attended beside the centroid tiles: the same blocks, so equal counts, and outputs that differ
    # from the one-block kernel's in the order of the sums only.
    print(f"early blocks: D{d} Tq{tq} Tk{tk} H{heads}", flush=True)
    q, k, v = (block_smooth(1, t, heads, d, seed=s, device="cuda") for t, s in ((tq, 1), (tk, 2), (tk, 3)))
    for local, beta in ((0, 1.0), (1, 1.0), (2, math.inf), (7, 0.0), (1 << 30, 1.0)):
        small, c0 = _launch(q, k, v, 0, monkeypatch, beta, local=local)
        one, c1 = _launch(q, k, v, 1, monkeypatch, beta, local=local)
        assert torch.equal(c0, c1)
        assert_close(small.cpu(), one.cpu())


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tq,tk,heads", [(121, 63, 3), (64, 64, 2), (75, 75, 3), (300, 128, 2), (300, 129, 2)])
def test_small_launches_of_one_or_two_key_blocks(d, tq, tk, heads, monkeypatch):
    # Two key-split groups at head_dim 128 up to two blocks, with fewer blocks than groups.
    print(f"short keys: D{d} Tq{tq} Tk{tk}", flush=True)
    q, k, v = tensors(tq, tk, d, 2, heads, device="cuda", seed=12)
    for local, beta in ((0, 1.0), (1, 0.0), (-1, math.inf)):
        small, c0 = _launch(q, k, v, 0, monkeypatch, beta, local=local)
        one, c1 = _launch(q, k, v, 1, monkeypatch, beta, local=local)
        assert torch.equal(c0, c1)
        assert_close(small.cpu(), one.cpu())


def _windows(kind, n):
    rows = torch.stack((torch.arange(0, 200), torch.arange(500, 700)))
    if kind == "runs":         # every whole block consecutive
        keys = torch.stack((torch.arange(0, 640), torch.arange(n - 640, n)))
    elif kind == "joined":     # blocks across a join are not
        keys = torch.stack((torch.cat((torch.arange(0, 100), torch.arange(300, 823))),
                            torch.cat((torch.arange(0, 100), torch.arange(1000, 1523)))))
    elif kind == "sparse":     # none is
        keys = torch.stack((torch.arange(0, 1200, 2), torch.arange(1, 1201, 2)))
    else:                      # ragged, with partial last blocks
        keys = [torch.arange(5, 705), torch.cat((torch.arange(0, 64), torch.arange(70, 400), torch.arange(900, 1111)))]
    return rows, keys


@pytest.mark.parametrize("d,h", [(64, 3), (128, 2), (128, 4)])
@pytest.mark.parametrize("kind", ["runs", "joined", "sparse", "ragged"])
@pytest.mark.parametrize("small", [True, False])
def test_windows_from_rows_equal_windows_from_tiles(d, h, kind, small, monkeypatch):
    print(f"windows: D{d} H{h} {kind} small {small}", flush=True)
    n = 1600
    gen = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((n, 2 * h, d), generator=gen).to(torch.bfloat16).cuda()[:, ::2] for _ in range(3))
    rows, keys = _windows(kind, n)
    plan = IndexedPlan.create(rows, keys, n, protected_ranges=((0, 7),), local_tokens=64).to("cuda")
    if not small:
        monkeypatch.setattr(_native, "WORKGROUP_FORM", 1)   # sol_attention_kernel, not the small kernel
    for beta in (-math.inf, 0.5, math.inf):
        got = sol_attention_indexed(q, k, v, plan, beta=beta)
        with monkeypatch.context() as mp:
            mp.setattr(_native, "_one_block_keys", lambda nk, d: False)
            assert torch.equal(got, sol_attention_indexed(q, k, v, plan, beta=beta))


CLASSES = 20


def _peaked(t, h, d, seed):
    """Q, K, V [t, h, d]: query i scores about 40 log2 units more against the
    keys of every 20th run of 32 than against the others.  So the max of some
    query of every wave jumps in nearly every half tile, and that half's scores are
    what its output is made of."""
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((t, h, d), generator=gen) for _ in range(3))
    peak = (40 * d ** 0.5 / math.log2(math.e)) ** 0.5
    i = torch.arange(t)
    q[i, :, i % CLASSES] += peak
    k[i, :, i // 32 % CLASSES] += peak
    return tuple(x.to(torch.bfloat16).cuda() for x in (q, k, v))


def _check_dense64(got, q, k, v, groups):
    """got [nq, h, d] against dense attention in 64 bits.  P and the output are
    rounded to BF16 (8 significant bits: by at most 2^-8 each, of at most sum
    p |v|), exponents and sums to FP32 (2^-11 together, generously).  Also that
    every key-split group meets half tiles whose row sum exceeds the lazy
    softmax's bound after the group's first tile."""
    d = q.shape[-1]
    for h in range(q.shape[1]):
        s = q[:, h].double() @ k[:, h].double().t().contiguous() * d ** -0.5
        p = torch.softmax(s, 1)
        vh = v[:, h].double()
        bound = (2 ** -7 + 2 ** -11) * (p @ vh.abs())
        err = (got[:, h].double() - p @ vh).abs()
        assert bool((err <= bound).all()), f"head {h}: {float((err / bound).max()):.2f} times the bound"
        if h == 0:
            s = s[:32] * math.log2(math.e)   # one wave's queries
            for g in range(groups):
                own = [t for j in range(g, -(-s.shape[1] // 64), groups) for t in (s[:, 64 * j:64 * j + 32],
                                                                                  s[:, 64 * j + 32:64 * j + 64])]
                m, jumps = torch.cat(own[:2], 1).amax(1), 0
                for half in own[2:]:
                    if half.shape[1] == 0:
                        continue
                    jumps += bool((torch.exp2(half - m[:, None]).sum(1) > 65535).any())
                    m = torch.maximum(m, half.amax(1))
                assert jumps >= 2 or len(own) < 8, f"group {g}: {jumps} jumps"


@pytest.mark.parametrize("d,h", [(64, 3), (128, 2), (64, 33), (128, 33)])   # four groups; two
@pytest.mark.parametrize("kind", ["runs", "joined", "sparse", "ragged"])
@pytest.mark.parametrize("form", [0, 1])
def test_jumping_scores_of_windows_equal_dense(d, h, kind, form, monkeypatch):
    print(f"jumping scores: D{d} H{h} {kind} form {form}", flush=True)
    n = 1600
    q, k, v = _peaked(n, h, d, seed=8)
    rows, keys = _windows(kind, n)
    plan = IndexedPlan.create(rows, keys, n, protected_ranges=((0, n),), local_tokens=0).to("cuda")
    monkeypatch.setattr(_native, "WORKGROUP_FORM", form)
    groups = 1 if form else (4 if 2 * 4 * h <= 256 else 2)
    for beta in (1.0, math.inf) if form == 0 else (1.0, -math.inf):
        got = sol_attention_indexed(q, k, v, plan, beta=beta)
        for w in range(2):
            kw = keys[w].cuda()
            _check_dense64(got[w], q[rows[w].cuda()], k[kw], v[kw], groups)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tk", [700, 2304, 4133])
@pytest.mark.parametrize("h", [2, 90])   # four groups; two
def test_jumping_scores_of_plain_keys_equal_dense(d, tk, h, monkeypatch):
    print(f"jumping scores: D{d} Tk{tk} H{h}", flush=True)
    q, k, v = _peaked(tk, h, d, seed=9)
    q = q[:150].contiguous()
    for form in (0, 1):
        got, _ = _launch(q[None], k[None], v[None], form, monkeypatch, 1.0, local=1 << 30)
        _check_dense64(got[0], q, k, v, 1 if form else (4 if 3 * h <= 256 else 2))


@pytest.mark.parametrize("d,h,copies", [(64, 2, 1), (128, 4, 1), (128, 4, 160)])
def test_block_rows(d, h, copies):
    # copies: enough windows for the four-head pooling kernel.
    n = 1600
    gen = torch.Generator().manual_seed(5)
    k, v = (torch.randn((n, h, d), generator=gen).to(torch.bfloat16).cuda() for _ in range(2))
    _, keys = _windows("joined", n)
    keys = keys.repeat(copies, 1)
    out = _native.pool_kv(k, v, key_index=keys.cuda(), windows=True)
    full = _native.pool_kv(k, v, key_index=keys.cuda())
    w, nk = keys.shape
    nkb = -(-nk // 64)
    off = out["block_rows_ptr"] - out["workspace"].data_ptr()
    got = out["workspace"][off:off + w * nkb * 4].view(torch.int32).view(w, nkb).cpu().numpy()
    kn = keys.numpy()
    want = np.full((w, nkb), -1)
    for j in range(nk // 64):
        blk = kn[:, 64 * j:64 * j + 64]
        run = (blk == blk[:, :1] + np.arange(64)).all(1)
        want[:, j] = np.where(run, blk[:, 0], -1)
    assert (want >= 0).any() and (want < 0).any()
    np.testing.assert_array_equal(got, want)
    assert torch.equal(out["ctiles"], full["ctiles"])
    for a in ("mean", "var"):
        assert torch.equal(out[a], full[a])
    copied = torch.from_numpy(want < 0).cuda()
    for b in range(w):
        assert torch.equal(out["tiles"][b, :, copied[b]], full["tiles"][b, :, copied[b]])


@pytest.mark.parametrize("kind", ["runs", "joined"])
def test_debug_launches_of_windows_hand_out_every_tile(kind):
    n, h, d = 1600, 2, 64
    gen = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn((n, h, d), generator=gen).to(torch.bfloat16).cuda() for _ in range(3))
    rows, keys = (x.cuda() for x in _windows(kind, n))
    out, _, dbg = _native.launch_sol(q, k, v, d ** -0.5, 1.0, -1, 0, 0, False, rows=rows, keys=keys, debug=True)
    assert torch.equal(dbg["tiles"], _native.pool_kv(k, v, key_index=keys)["tiles"])
    plain, _ = _native.launch_sol(q, k, v, d ** -0.5, 1.0, -1, 0, 0, False, rows=rows, keys=keys)
    assert torch.equal(out, plain)
