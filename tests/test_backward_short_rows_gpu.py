"""dQ of queries that see at most 1152 keys, computed in half-size workgroups in steps of 32 columns: for the
windows the same products in the same order as in the large ones, so the same bits."""
import pytest
import torch

from plan_util import backward
from test_backward_gpu import kernel_grads, make, run_case

pytestmark = pytest.mark.gpu
LIMIT = 1152  # keys up to which a row is short
HEADS = [(2, 2), (4, 2), (8, 2)]  # 1, 2 and 4 heads of a kv head in one workgroup


@pytest.mark.parametrize("H,Hkv", HEADS)
@pytest.mark.parametrize("S", [1, 31, 32, 33, 63, 64, 65, 127, 129, 1000, LIMIT, 1500])
def test_same_bits_in_either_size(monkeypatch, S, H, Hkv):
    """INTRA_WAVES names the size; unnamed, the limit decides."""
    q, k, v, dout = make(2, S, H, Hkv, seed=S)
    grads = {}
    for waves in (8, 4):
        monkeypatch.setenv("INTRA_WAVES", str(waves))
        assert backward("window", 2, S, H, Hkv, window=300)[0].waves == waves
        grads[waves] = kernel_grads(q, k, v, dout, "window", window=300)
    for name, a, b in zip(("dq", "dk", "dv"), grads[8], grads[4]):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("H,Hkv", HEADS)
@pytest.mark.parametrize("S", [33, 129, 1000, 1500])
@pytest.mark.parametrize("waves", [8, 4])
def test_windows_with_sinks_in_either_size(monkeypatch, waves, S, H, Hkv):
    """The columns of a row block start where its first query's window does, so the sizes share no blocks of 32."""
    monkeypatch.setenv("INTRA_WAVES", str(waves))
    assert backward("window_sink", 1, S, H, Hkv, window=300, n_sink=33)[0].waves == waves
    run_case("llm/window_sink", "window_sink", 1, S, H, Hkv, window=300, n_sink=33)


@pytest.mark.parametrize("H,Hkv", HEADS)
@pytest.mark.parametrize("columns", [LIMIT - 1, LIMIT, LIMIT + 1])
def test_grads_at_the_limit(columns, H, Hkv):
    assert backward("window", 1, 2300, H, Hkv, window=columns)[0].waves == (4 if columns <= LIMIT else 8)
    run_case("llm/window", "window", 1, 2300, H, Hkv, window=columns)
    run_case("llm/window_sink", "window_sink", 1, 2300, H, Hkv, window=columns - 33, n_sink=33)
