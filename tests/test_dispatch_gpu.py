"""Every row of every head, O and the natural-log L, for sizes on both sides of the rules
that choose a kernel or a work order by problem size."""

import pytest
import torch

from helpers import FWD_ATOL, max_abs, oracle_fwd, randn

pytestmark = pytest.mark.gpu


def check_forward(B, Hq, Hkv, Nq, Nk, d, causal):
    from flash_attn_legacy import hip_ext
    q, k, v = randn((B, Hq, Nq, d), 0), randn((B, Hkv, Nk, d), 1), randn((B, Hkv, Nk, d), 2)
    scale = d ** -0.5
    o, lse = hip_ext.forward(q, k, v, scale, causal)
    ref_o, ref_l = oracle_fwd(q, k, v, scale, causal)
    assert torch.isfinite(o).all()
    assert max_abs(o, ref_o) <= FWD_ATOL
    assert max_abs(lse, ref_l) <= FWD_ATOL


# Causal grids by workgroup count (128 query rows each): two per CU at most (264, 348), more
# (704, 675, and 288 at one per CU for head_dim 256); heads that divide by 8 and that do not;
# a last tile of one row.
@pytest.mark.parametrize("B,Hq,Hkv,N,d", [
    (8, 11, 11, 300, 64),
    (3, 29, 29, 400, 64),
    (8, 22, 11, 385, 32),
    (5, 27, 9, 520, 96),
    (4, 24, 8, 300, 256),
])
def test_causal_order(B, Hq, Hkv, N, d):
    check_forward(B, Hq, Hkv, N, N, d, True)
