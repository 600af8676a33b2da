"""The order in which a launch deals its work items depends on its size (row block by row block where pair by pair
would leave some workgroups with much more than the others); the results do not.  A call on one kv head and its
query heads has one pair per XCD at most, so only one order: a call on all heads has to give the same bits."""
import os

import pytest
import torch

from intra_amd import intra_llm_attn
from parity_util import make_qkv
from plan_util import forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", ["8", "4"])
@pytest.mark.parametrize("pattern,B,S,H,Hkv,kw", [
    ("scatter", 1, 5000, 32, 8, dict(group_num=8)),   # 10 row blocks of 8 pairs per XCD
    ("scatter", 1, 7001, 28, 4, dict(group_num=3)),   # 7 query heads of a kv head one by one, 1 or 2 pairs per XCD
    ("block_scatter", 1, 6000, 32, 8, dict(group_num=2, block=256, offset=1, n_sink=64)),
    ("window", 2, 5000, 32, 8, dict(window=2112)),
    ("gather1", 1, 4992, 16, 8, dict(group_num=8)),
])
def test_same_bits_in_either_order(monkeypatch, waves, pattern, B, S, H, Hkv, kw):
    monkeypatch.setitem(os.environ, "INTRA_WAVES", waves)
    q, k, v = make_qkv(B, S, H, Hkv, seed=S)
    r = H // Hkv
    assert forward(pattern, B, S, H, Hkv, **kw).row_order == 1 and forward(pattern, 1, S, r, 1, **kw).row_order == 0
    with torch.no_grad():
        out = intra_llm_attn(q, k, v, pattern, **kw)
        for h in range(Hkv):
            one = intra_llm_attn(q[:1, :, h * r:(h + 1) * r], k[:1, :, h:h + 1], v[:1, :, h:h + 1], pattern, **kw)
            assert torch.equal(out[:1, :, h * r:(h + 1) * r], one), (pattern, h)
