"""Which workgroup form a launch takes (one or two query blocks per workgroup), by the library's own rule.

No counterpart in the reference (one Triton program per query block).
"""

import math
import os

import pytest

from sol_attn_amd import _native

pytestmark = pytest.mark.skipif(not os.path.exists(_native.LIB_PATH), reason="libsol_attn_amd.so not built")


@pytest.mark.parametrize("b,nq,nk,h,d,int8,one", [
    # INT8 scores have a two-slot ring in either form: two blocks, as half the waves fit otherwise.
    (2, 4096, 4096, 16, 128, False, True), (2, 4096, 4096, 16, 128, True, False),
    (1, 16384, 16384, 8, 128, True, False),
    (2, 4096, 4096, 16, 64, True, False),
    (1, 4096, 4096, 4, 128, True, True),       # 128 pairs: two blocks would leave CUs idle
])
def test_int8_launches(b, nq, nk, h, d, int8, one):
    assert _native._one_block(b, nq, nk, h, d, 1.0, int8, False) == one


def test_int8_launches_pair_their_query_blocks():
    # 8,192 query blocks and more.
    assert _native._pairs(1, 32768, 24000, 24, 128, 1.0, True, False)
    assert not _native._windows(21, 4032, 8064, 24, 128, 1.0, True)
    assert not _native._windows(2, 1823, 3646, 32, 64, 1.0, True) and _native._windows(2, 1823, 3646, 32, 64, 1.0, False)
    assert _native._windows(8, 1000, 4000, 2, 64, 1.0, True)   # fewer than 512 pairs


@pytest.mark.parametrize("b,nq,nk,h,d,beta,windows,one", [
    # At most half the key blocks selected, and these at most half the query blocks.
    (2, 4096, 4096, 16, 128, 0.0, False, True), (2, 4096, 4096, 16, 128, -0.1, False, False),
    (2, 4096, 4096, 16, 128, -math.inf, False, False), (2, 4096, 4096, 16, 128, math.inf, False, True),
    (1, 4096, 10000, 24, 128, 1.0, False, True), (1, 4096, 10000, 24, 128, 0.0, False, False),
    (1, 2048, 16384, 32, 128, 1.0, False, False), (1, 8192, 1000, 16, 64, -1.0, False, False),
    # K and V at most 12 MB per head.
    (1, 24576, 24576, 24, 128, 1.0, False, True), (1, 24577, 24577, 24, 128, 1.0, False, False),
    (1, 49152, 49152, 24, 64, 1.0, False, True), (1, 49153, 49153, 24, 64, math.inf, False, False),
    # 5 MB of them selected.
    (1, 24576, 24576, 24, 128, 0.0, False, False), (1, 20000, 20000, 24, 128, 0.0, False, True),
    # Windows: 70% selected, or at most 192 key blocks.
    (21, 4032, 16128, 24, 128, -0.5, True, True), (21, 4032, 16128, 24, 128, -1.0, True, False),
    (21, 3000, 12000, 24, 128, -math.inf, True, True), (21, 4032, 16128, 24, 128, -math.inf, True, False),
    # Fewer than 512 pairs of query blocks.
    (1, 4096, 100000, 15, 128, -math.inf, False, True),
])
def test_selected_share_and_key_bytes(b, nq, nk, h, d, beta, windows, one):
    assert _native._one_block(b, nq, nk, h, d, beta, False, windows) == one


def test_dense_selections_pair_their_query_blocks():
    assert _native._pairs(1, 24576, 24576, 24, 128, -1.0, False, False)
    assert not _native._pairs(1, 24576, 24576, 24, 128, 1.0, False, False)
    assert not _native._pairs(21, 4032, 12096, 24, 128, 0.0, False, True)
