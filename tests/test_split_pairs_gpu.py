"""Where the (set, batch, kv head) pairs of a call do not come out even over the XCDs, the row blocks of a pair are
split over several of them (xcd_split).  Eight kv heads come out even, one to three of them do not: the same bits."""
import os

import pytest
import torch

import oracle
from intra_amd import _lib, intra_llm_attn, intra_llm_attn_bwd
from plan_util import backward, backward_of, forward
from test_backward_gpu import DEV, compare, make

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

    def parts(n):  # of the forward and of the backward's launches
        return [x.parts for x in (forward(pattern, 1, S, n * r, n, **kw), *backward(pattern, 1, S, n * r, n, **kw))]

    assert max(parts(8)) == 1
    want = run(q, k, v, dout)
    for first, n in ((0, 1), (1, 2), (3, 3), (2, 5)):
        heads, kv = slice(first * r, (first + n) * r), slice(first, first + n)
        assert n == 5 or max(parts(n)) > 1
        got = run(q[:, :, heads], k[:, :, kv], v[:, :, kv], dout[:, :, heads])
        for name, a, b, at in zip(("out", "lse", "dq", "dk", "dv"), got, want, (heads, heads, heads, kv, kv)):
            b = b[:, at] if name == "lse" else b[:, :, at]
            if name in ("dk", "dv"):  # (the sinks' gradients are added up in chunks, fewer for more heads)
                a, b = a[:, kw.get("n_sink", 0):], b[:, kw.get("n_sink", 0):]
            assert torch.equal(a, b), (name, first, n)


@pytest.mark.parametrize("pattern,pid", [("scatter", 0), ("gather0", 4)])
def test_text_keys_of_an_image_in_parts(pattern, pid):
    """A text so long that its keys are more row blocks than the device has CUs, on nine heads (through the C ABI: the
    public calls have 512 text tokens, which always fit one round)."""
    lib, width, text_len, H, scale = _lib.load(), 16, 4224, 9, 128 ** -0.5
    shape = (1, text_len + width * width, H, H)
    assert [x.parts for x in backward_of(1, pid, *shape, width, text_len, 0, 0, 0) if x.keys and x.leading] == [2]
    q, k, v, dout = make(*shape, seed=9)
    stream = torch.cuda.current_stream().cuda_stream
    out, lse = torch.empty_like(q), torch.empty(1, H, shape[1], dtype=torch.float32, device=DEV)
    rc = lib.intra_image_fwd_lse(*(x.data_ptr() for x in (q, k, v, out)), *shape, *(_lib.strides3(x) for x in (q, k, v, out)),
                                 pid, width, text_len, scale, stream, lse.data_ptr(), _lib.strides3(lse))
    assert rc == 0, _lib.last_error()
    work = torch.empty(lib.intra_image_bwd_workspace(*shape, pid, width, text_len), dtype=torch.float32, device=DEV)
    got = tuple(torch.full_like(t, float("nan")) for t in (q, k, v))
    rc = lib.intra_image_bwd(*(x.data_ptr() for x in (q, k, v, out, lse, dout, *got, work)), *shape,
                             *(_lib.strides3(x) for x in (q, k, v, out, dout, *got, lse)), pid, width, text_len, scale, stream)
    assert rc == 0, _lib.last_error()
    mask = oracle.mask_rows(f"image/{pattern}", shape[1], device=DEV, width=width, text_len=text_len)
    compare(got, oracle.masked_attention_grads(q, k, v, dout, mask), f"image/{pattern} T={text_len}")
