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
