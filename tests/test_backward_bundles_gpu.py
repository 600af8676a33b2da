"""The order in which a backward launch starts its workgroups depends on its size (all pairs of an XCD together where
the longest row blocks of a last bundle would start late); the results do not.  A call on one kv head and its query
heads has one pair per XCD at most: a call on all heads has to give the same bits."""
import pytest
import torch

from intra_amd import intra_llm_attn, intra_llm_attn_bwd
from plan_util import backward, one_bundle
from test_backward_gpu import make

pytestmark = pytest.mark.gpu


# together: the launches (dQ, dK / dV) that take all pairs of an XCD as one bundle
@pytest.mark.parametrize("pattern,B,S,H,Hkv,kw,sets,together", [
    ("scatter", 1, 7000, 32, 8, dict(group_num=3), 3, [True, True]),
    ("scatter", 1, 3000, 16, 16, dict(group_num=4), 4, [False, True]),
    ("scatter", 2, 2501, 8, 8, dict(group_num=4), 4, [False, True]),
    ("gather1", 1, 4992, 16, 8, dict(group_num=8), 8, [True, True]),
    ("block_scatter", 1, 6000, 16, 16, dict(group_num=2, block=256, offset=0, n_sink=0), 2, [True, False]),
    ("window", 4, 1700, 8, 8, dict(window=1600), 1, [False, True]),
])
def test_same_bits_in_either_order(pattern, B, S, H, Hkv, kw, sets, together):
    q, k, v, dout = make(B, S, H, Hkv, seed=S)
    r = H // Hkv
    assert [one_bundle(rows, B * Hkv * sets) for rows in backward(pattern, B, S, H, Hkv, **kw)] == together
    assert not any(one_bundle(rows, sets) for rows in backward(pattern, 1, S, r, 1, **kw))

    def grads(*tensors):
        with torch.no_grad():
            out, lse = intra_llm_attn(*tensors[:3], pattern, return_lse=True, **kw)
            return intra_llm_attn_bwd(*tensors[:3], out, lse, tensors[3], pattern, **kw)

    got = grads(q, k, v, dout)
    for h in (0, Hkv // 2, Hkv - 1):
        one = grads(*(x[-1:, :, h * n:(h + 1) * n] for x, n in ((q, r), (k, 1), (v, 1), (dout, r))))
        for name, a, b, n in zip(("dq", "dk", "dv"), got, one, (r, 1, 1)):
            assert torch.equal(a[-1:, :, h * n:(h + 1) * n], b), (name, h)
