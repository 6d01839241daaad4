"""Which workgroup form a launch takes (one or two query blocks per workgroup), by the library's own rule.

No counterpart in the reference (one Triton program per query block).
"""

import os

import pytest

from sol_attn_amd import _native

pytestmark = pytest.mark.skipif(not os.path.exists(_native.LIB_PATH), reason="libsol_attn_amd.so not built")


@pytest.mark.parametrize("b,nq,nk,h,d,int8,one", [
    # INT8 scores at head_dim 128 have a two-slot ring in either form: two blocks, as half the waves fit otherwise.
    (2, 4096, 4096, 16, 128, False, True), (2, 4096, 4096, 16, 128, True, False),
    (1, 16384, 16384, 8, 128, True, False),
    (2, 4096, 4096, 16, 64, True, True),
    (1, 4096, 4096, 4, 128, True, True),       # 128 pairs: two blocks would leave CUs idle
])
def test_int8_launches(b, nq, nk, h, d, int8, one):
    assert _native._one_block(b, nq, nk, h, d, int8) == one


def test_int8_launches_pair_their_query_blocks():
    # 8,192 query blocks and more.
    assert _native._pairs(1, 32768, 24000, 24, 128, True)
    assert not _native._windows(21, 4032, 8064, 24, 128, True)
