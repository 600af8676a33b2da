"""What a call of intra_amd's entry points launches (host only, counted for 256 CUs): so that tests of one route
can say that the call takes it."""
import ctypes

from intra_amd import _lib
from intra_amd.interface import EXTRA_LLM_PATTERNS, LLM_PATTERNS

LLM = 0
IDS = dict(LLM_PATTERNS, **EXTRA_LLM_PATTERNS)


def _args(pattern, B, S, H, Hkv, group_num=8, window=576, block=256, offset=0, n_sink=0):
    return LLM, IDS[pattern], B, S, H, Hkv, group_num, window, block, offset, n_sink


def backward(pattern, B, S, H, Hkv, **kw):
    """The kinds of rows of the backward's launches, in order: queries (dq), keys, leading keys."""
    return backward_of(*_args(pattern, B, S, H, Hkv, **kw))


def backward_of(*args):
    rows, n = (_lib.IntraBwdRows * 5)(), ctypes.c_int()
    rc = _lib.load().intra_plan_bwd(*args, rows, 5, ctypes.byref(n))
    assert rc == 0, _lib.last_error()
    return rows[:n.value]


def one_bundle(rows, pairs):
    """Whether an XCD's (set, batch, kv head) pairs are worked on together where fewer of them would fill its CUs"""
    per_xcd = -(-pairs * rows.parts // 8)
    places = 32 if rows.waves == 8 or rows.keys else 64
    return rows.bundle == per_xcd > -(-places // (rows.row_blocks * rows.head_groups))


def forward(pattern, B, S, H, Hkv, **kw):
    """Order in which the forward's row blocks are dealt"""
    deal = _lib.IntraDeal()
    assert _lib.load().intra_plan_deal(*_args(pattern, B, S, H, Hkv, **kw), deal) == 0, _lib.last_error()
    return deal
