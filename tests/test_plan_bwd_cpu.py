"""Which workgroups a backward call launches (intra_plan_bwd, host only): the sizes of dQ's workgroups and the split
of few pairs' row blocks over the XCDs."""
import ctypes

import pytest

from intra_amd import _lib
from plan_util import backward_of

LLM, IMAGE = 0, 1
SCATTER, WINDOW, GATHER0, BLOCK_SCATTER, WINDOW_SINK = 0, 4, 4, 8, 9
XCDS, CUS = 8, 32


def plan(domain, pattern, B, S, H, Hkv, arg0=0, arg1=0, block=64, offset=0, n_sink=0):
    return backward_of(domain, pattern, B, S, H, Hkv, arg0, arg1, block, offset, n_sink)


def window(B, S, H, Hkv, width, n_sink=None):
    if n_sink is None:
        return plan(LLM, WINDOW, B, S, H, Hkv, 8, width)
    return plan(LLM, WINDOW_SINK, B, S, H, Hkv, 8, width, n_sink=n_sink)


def test_entries_are_the_kinds_of_rows_of_a_call():
    kinds = lambda rows: [(r.keys, r.leading) for r in rows]
    assert kinds(plan(LLM, SCATTER, 1, 4096, 32, 8, 8)) == [(0, 0), (1, 0)]
    assert kinds(window(1, 4096, 32, 8, 575, n_sink=64)) == [(0, 0), (1, 0), (1, 1)]
    assert kinds(plan(IMAGE, GATHER0, 1, 4608, 24, 24, 64, 512)) == [(0, 0), (0, 1), (1, 0), (1, 1), (1, 0)]
    rows, n = (_lib.IntraBwdRows * 1)(), ctypes.c_int()
    lib = _lib.load()
    assert lib.intra_plan_bwd(LLM, SCATTER, 1, 4096, 32, 8, 8, 0, 0, 0, 0, rows, 1, ctypes.byref(n)) == 0 and n.value == 2
    assert lib.intra_plan_bwd(LLM, BLOCK_SCATTER, 1, 512, 4, 4, 2, 0, 64, 1, 0, rows, 1, ctypes.byref(n)) == _lib.INTRA_ERR_UNSUPPORTED
    assert lib.intra_plan_bwd(LLM, SCATTER, 1, 4096, 32, 8, 8, 0, 0, 0, 0, None, 1, ctypes.byref(n)) == _lib.INTRA_ERR_INVALID


@pytest.mark.parametrize("n_sink", [None, 64])
@pytest.mark.parametrize("S,H,Hkv", [(8000, 4, 1), (2000, 8, 1), (4000, 4, 1), (4000, 8, 2), (3000, 8, 2), (2048, 4, 1)])
def test_half_size_workgroups_take_a_cu_each_before_they_share_one(S, H, Hkv, n_sink):
    """As many row blocks as the CUs of some XCDs hold one by one, or fewer: none of these XCDs gets a 33rd."""
    dq = window(1, S, H, Hkv, 576, n_sink)[0]
    assert dq.keys == 0 and dq.waves == 4
    per_pair = -(-S // dq.rows_per_block) * dq.head_groups
    assert per_pair * Hkv <= XCDS * CUS
    fullest = -(-Hkv * dq.parts // XCDS) * dq.row_blocks * dq.head_groups
    assert fullest <= CUS, (dq.parts, dq.row_blocks, fullest)


@pytest.mark.parametrize("S,width,waves", [
    (1000, 576, 4), (1000, 4096, 4), (1152, 4096, 4), (1153, 4096, 8), (3000, 1152, 4), (3000, 1153, 8), (700, 2 ** 31 - 1, 4)])
def test_short_rows_are_those_of_queries_that_see_few_keys(S, width, waves):
    """Up to 1152 keys, of those that there are: a window longer than the sequence is as long as the sequence."""
    assert window(1, S, 8, 2, width)[0].waves == waves
    assert window(1, S, 8, 2, width, n_sink=0)[0].waves == waves
    if S >= 1153 and width >= 1152:
        assert window(1, S, 8, 2, width - 33, n_sink=33)[0].waves == waves


# dQ of image Gather 0: half-size workgroups where the fullest of the CUs then gets less to do (or as much, in more than
# one round, and each less of the tiles)
@pytest.mark.parametrize("width,B,H,Hkv,waves", [
    (64, 1, 3, 3, 4), (64, 1, 6, 6, 4), (64, 1, 12, 12, 8), (64, 2, 6, 6, 8), (64, 1, 16, 16, 4), (64, 1, 24, 24, 4),
    (64, 1, 8, 4, 8), (64, 1, 24, 6, 8), (64, 1, 16, 4, 4), (128, 1, 3, 3, 8), (128, 1, 6, 6, 4), (128, 1, 12, 12, 4),
    (128, 1, 24, 24, 4), (128, 1, 8, 4, 4), (128, 1, 4, 1, 4)])
def test_gather0_dq_workgroups_follow_the_rounds(width, B, H, Hkv, waves):
    patches, text = plan(IMAGE, GATHER0, B, 512 + width * width, H, Hkv, width, 512)[:2]
    assert (patches.keys, text.keys, text.leading) == (0, 0, 1)
    assert patches.waves == text.waves == waves
    assert patches.rows_per_block == text.rows_per_block == waves * 32 // (H // Hkv)


def test_text_keys_of_an_image_can_be_split_too():
    """33 row blocks of text keys for 9 heads: more workgroups than CUs, so the queries are one chunk and the 9 pairs
    leave XCDs with a third round; the public calls (512 text keys) always fit one round."""
    for pattern in (SCATTER, GATHER0):
        text = [r for r in plan(IMAGE, pattern, 1, 4224 + 256, 9, 9, 16, 4224) if r.keys and r.leading]
        assert [r.parts for r in text] == [2]
        for width, B, H in ((64, 1, 3), (64, 1, 24), (64, 3, 40), (128, 1, 5), (128, 2, 24)):
            assert all(r.parts == 1 for r in plan(IMAGE, pattern, B, 512 + width * width, H, H, width, 512))


@pytest.mark.parametrize("Hkv", [8, 16, 32])
def test_pairs_that_come_out_even_stay_whole(Hkv):
    for rows in (window(1, 5000, Hkv, Hkv, 576), plan(LLM, SCATTER, 1, 5000, Hkv, Hkv, 8)):
        assert [r.parts for r in rows] == [1, 1]
