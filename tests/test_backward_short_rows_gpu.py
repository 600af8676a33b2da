"""dQ of row blocks that meet at most 1152 columns, computed in half-size workgroups in steps of 32 columns: the same
products in the same order as in the large ones, so the same bits."""
import pytest
import torch

from test_backward_gpu import kernel_grads, make, run_case

pytestmark = pytest.mark.gpu
LIMIT = 1152  # columns up to which a row block is short
HEADS = [(2, 2), (4, 2), (8, 2)]  # 1, 2 and 4 heads of a kv head in one workgroup


@pytest.mark.parametrize("H,Hkv", HEADS)
@pytest.mark.parametrize("S", [1, 31, 32, 33, 63, 64, 65, 127, 129, 1000, LIMIT])
def test_same_bits_on_both_sides_of_the_limit(S, H, Hkv):
    """Windows that no sequence of S tokens fills are one mask."""
    q, k, v, dout = make(2, S, H, Hkv, seed=S)
    short = kernel_grads(q, k, v, dout, "window", window=LIMIT)
    long = kernel_grads(q, k, v, dout, "window", window=LIMIT + 1)
    for name, a, b in zip(("dq", "dk", "dv"), short, long):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("H,Hkv", HEADS)
@pytest.mark.parametrize("columns", [LIMIT - 1, LIMIT, LIMIT + 1])
def test_grads_at_the_limit(columns, H, Hkv):
    run_case("llm/window", "window", 1, 2300, H, Hkv, window=columns)
    run_case("llm/window_sink", "window_sink", 1, 2300, H, Hkv, window=columns - 33, n_sink=33)
