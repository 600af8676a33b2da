"""Where the (set, batch, kv head) pairs of a call do not come out even over the XCDs, the row blocks of a pair are
split over several of them (xcd_split).  Eight kv heads come out even, one to three of them do not: the same bits."""
import os

import pytest
import torch

from intra_amd import intra_llm_attn, intra_llm_attn_bwd
from test_backward_gpu import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", ["8", "4"])
@pytest.mark.parametrize("pattern,S,r,kw", [
    ("window", 4997, 1, dict(window=1000)),                # 40 key blocks, 20 query blocks
    ("window", 5000, 4, dict(window=300)),                 # the forward's and dQ's row blocks are of 64 queries
    ("window_sink", 4500, 2, dict(window=200, n_sink=70)),
    ("window_sink", 6111, 1, dict(window=1500, n_sink=4)),
    ("scatter", 13001, 4, dict(group_num=3)),
    ("block_scatter", 9001, 4, dict(group_num=2, block=256, offset=1, n_sink=64)),
])
def test_same_bits_for_few_kv_heads(monkeypatch, waves, pattern, S, r, kw):
    monkeypatch.setitem(os.environ, "INTRA_WAVES", waves)
    q, k, v, dout = make(1, S, 8 * r, 8, seed=S)

    def run(*tensors):
        with torch.no_grad():
            out, lse = intra_llm_attn(*tensors[:3], pattern, return_lse=True, **kw)
            return (out, lse, *intra_llm_attn_bwd(*tensors[:3], out, lse, tensors[3], pattern, **kw))

    want = run(q, k, v, dout)
    for first, n in ((0, 1), (1, 2), (3, 3), (2, 5)):
        heads, kv = slice(first * r, (first + n) * r), slice(first, first + n)
        got = run(q[:, :, heads], k[:, :, kv], v[:, :, kv], dout[:, :, heads])
        for name, a, b, at in zip(("out", "lse", "dq", "dk", "dv"), got, want, (heads, heads, heads, kv, kv)):
            b = b[:, at] if name == "lse" else b[:, :, at]
            if name in ("dk", "dv"):  # (the sinks' gradients are added up in chunks, fewer for more heads)
                a, b = a[:, kw.get("n_sink", 0):], b[:, kw.get("n_sink", 0):]
            assert torch.equal(a, b), (name, first, n)
