"""dQ of image Gather 0 in workgroups of 8 and of 4 wavefronts (INTRA_WAVES names the size), which split the patches
and the text rows into other row blocks: each against the oracle, and a plain call gives one of the two."""
import pytest
import torch

import oracle
from intra_amd import _lib
from test_backward_gpu import DEV, compare, make

pytestmark = pytest.mark.gpu
GATHER0 = 4


@pytest.mark.parametrize("H,Hkv", [(3, 3), (4, 2), (4, 1)])  # 1, 2 and 4 heads of a kv head in one workgroup
@pytest.mark.parametrize("width,text_len", [(16, 8), (24, 100 * 8), (40, 64), (64, 512), (72, 256)])
def test_both_sizes(monkeypatch, width, text_len, H, Hkv):
    lib, B, S, scale = _lib.load(), 2, text_len + width * width, 128 ** -0.5
    q, k, v, dout = make(B, S, H, Hkv, seed=width)
    stream = torch.cuda.current_stream().cuda_stream
    out, lse = torch.empty_like(q), torch.empty(B, H, S, dtype=torch.float32, device=DEV)
    shape = (B, S, H, Hkv)
    rc = lib.intra_image_fwd_lse(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), *shape,
                                 *(_lib.strides3(x) for x in (q, k, v, out)), GATHER0, width, text_len, scale, stream,
                                 lse.data_ptr(), _lib.strides3(lse))
    assert rc == 0, _lib.last_error()
    work = torch.empty(lib.intra_image_bwd_workspace(*shape, GATHER0, width, text_len), dtype=torch.float32, device=DEV)

    def grads(waves):
        if waves:
            monkeypatch.setenv("INTRA_WAVES", str(waves))
        else:
            monkeypatch.delenv("INTRA_WAVES", raising=False)
        got = tuple(torch.full_like(t, float("nan")) for t in (q, k, v))
        rc = lib.intra_image_bwd(*(x.data_ptr() for x in (q, k, v, out, lse, dout, *got, work)), *shape,
                                 *(_lib.strides3(x) for x in (q, k, v, out, dout, *got, lse)), GATHER0, width, text_len,
                                 scale, stream)
        assert rc == 0, _lib.last_error()
        return got

    mask = oracle.mask_rows("image/gather0", S, device=DEV, width=width, text_len=text_len)
    want = oracle.masked_attention_grads(q, k, v, dout, mask)
    by_size = [grads(8), grads(4)]
    for waves, got in zip((8, 4), by_size):
        compare(got, want, f"W={width} T={text_len} waves={waves}")
    plain = grads(None)
    assert any(all(torch.equal(a, b) for a, b in zip(plain, got)) for got in by_size)
