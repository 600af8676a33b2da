"""The dealing of work items to the persistent workgroups, enumerated on the host with the kernels' own
code (intra_model_deal): whatever the grid and the workgroup size, every row block that exists is
dealt exactly once - also where the heavy text row blocks of image gather0 stand for several rounds
of their workgroups - and no workgroup count changes which row blocks exist."""
import numpy as np
import pytest

from intra_amd import _lib

LLM, IMAGE = 0, 1
SCATTER, GATHER1, GATHER0, WINDOW = 0, 1, 4, 4


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def set_sizes(plan, domain, pattern, S, arg0, arg1):
    """Queries of every set, from what the patterns are (the text rows of image Gather 0 come first)."""
    if domain == IMAGE:
        chunk, grid = arg1 // 8, arg0 * arg0
        if pattern == SCATTER:
            return [chunk + grid // 8] * 8
        run = max(n for n in (1, 2, 4) if 64 * n <= plan.pos_per_block and arg0 // 8 % n == 0)  # patches
        n_text = plan.n_sets - grid // 64 // run
        assert n_text in (4, 8)
        return [8 // n_text * chunk] * n_text + [64 * run] * (grid // 64 // run)
    if pattern == WINDOW and arg1:
        return [S]
    token_group = (lambda t: t % arg0) if pattern == SCATTER else (lambda t: t // arg0 % arg0)
    return np.bincount(token_group(np.arange(S)), minlength=arg0).tolist()


class Dealing:
    """What the workgroups of a grid are dealt, and what they should be."""

    def __init__(self, lib, monkeypatch, waves, domain, pattern, B, S, H, Hkv, arg0, arg1):
        self.lib, self.call, self.waves = lib, (domain, pattern, B, S, H, Hkv, arg0, arg1), waves
        monkeypatch.setenv("INTRA_WAVES", str(waves))
        self.plan = plan = _lib.IntraPlan()
        assert lib.intra_plan(*self.call, plan) == 0, _lib.last_error()
        assert plan.waves == waves
        sizes = set_sizes(plan, domain, pattern, S, arg0, arg1)
        assert len(sizes) == plan.n_sets and -(-max(sizes) // plan.pos_per_block) == plan.n_mblocks
        real = np.arange(plan.n_mblocks) * plan.pos_per_block < np.array(sizes)[:, None]  # (set, row block)
        groups = H // Hkv // plan.heads_per_block
        self.expected = np.zeros(plan.work_items, dtype=np.uint8)
        items = np.broadcast_to(real[:, None, :, None], (plan.n_sets, B * Hkv, plan.n_mblocks, groups))
        self.expected[:items.size] = items.reshape(-1)

    def visits(self, grid):
        """None where there are fewer row blocks than workgroups."""
        visits = np.zeros(self.plan.work_items, dtype=np.uint8)
        rc = self.lib.intra_model_deal(*self.call, self.waves, grid, visits.ctypes.data, visits.size)
        if grid > self.plan.work_items:
            assert rc != 0 and "grid" in _lib.last_error()
            return None
        assert rc == 0, _lib.last_error()
        return visits

    def route(self):
        """(parts, row order) of the launch on 256 CUs"""
        deal = _lib.IntraDeal()
        assert self.lib.intra_plan_deal(*self.call, 0, 0, 0, deal) == 0, _lib.last_error()
        assert deal.waves == self.waves
        return deal.parts, deal.row_order

    def check(self, grids=(8, 16, 64, 256, 512, 1024)):
        for grid in grids:
            visits = self.visits(grid)
            assert visits is None or np.array_equal(visits, self.expected), (self.call, self.waves, grid)


@pytest.mark.parametrize("waves", [8, 4])
@pytest.mark.parametrize("width,B,H", [(64, 1, 24), (128, 1, 24), (128, 2, 24), (32, 1, 3), (96, 1, 5), (128, 1, 40)])
def test_image_gather0_every_row_block_once(lib, monkeypatch, width, B, H, waves):
    Dealing(lib, monkeypatch, waves, IMAGE, GATHER0, B, 512 + width * width, H, H, width, 512).check()


@pytest.mark.parametrize("waves", [8, 4])
@pytest.mark.parametrize("case", [
    (LLM, SCATTER, 1, 8192, 32, 8, 8, 0), (LLM, GATHER1, 2, 4100, 8, 2, 8, 0), (LLM, WINDOW, 1, 8192, 32, 8, 8, 576),
    (IMAGE, SCATTER, 1, 4608, 24, 24, 64, 512), (IMAGE, SCATTER, 1, 16896, 24, 24, 128, 512)])
def test_other_patterns_every_row_block_once(lib, monkeypatch, case, waves):
    dealing = Dealing(lib, monkeypatch, waves, *case)
    dealing.check()
    parts, row_order = dealing.route()
    assert parts == 1 and (case[0] == LLM or row_order == 0)


# Sizes whose pairs do not end with a round of the workgroups: dealt row block by row block where that is
# better balanced (which depends on the workgroup size)
@pytest.mark.parametrize("waves", [8, 4])
@pytest.mark.parametrize("case,row_order", [
    ((LLM, SCATTER, 1, 30000, 32, 8, 8, 0), {8: 1, 4: 1}), ((LLM, SCATTER, 1, 5000, 32, 8, 8, 0), {8: 1, 4: 1}),
    ((LLM, SCATTER, 1, 20000, 28, 4, 3, 0), {8: 1, 4: 1}), ((LLM, SCATTER, 3, 3000, 32, 8, 4, 0), {8: 1, 4: 1}),
    ((LLM, GATHER1, 1, 20032, 16, 8, 8, 0), {8: 1, 4: 1}), ((LLM, WINDOW, 2, 5000, 32, 8, 8, 2112), {8: 1, 4: 1}),
    ((LLM, SCATTER, 1, 2100, 8, 1, 9, 0), {8: 0, 4: 0})])
def test_uneven_sizes_every_row_block_once(lib, monkeypatch, case, row_order, waves):
    dealing = Dealing(lib, monkeypatch, waves, *case)
    dealing.check()
    assert dealing.route()[1] == row_order[waves]


@pytest.mark.parametrize("waves", [8, 4])
@pytest.mark.parametrize("pattern,arg0,arg1", [(SCATTER, 1, 0), (SCATTER, 3, 0), (WINDOW, 8, 576)])
@pytest.mark.parametrize("B,S,H,Hkv", [(1, 13568, 4, 1), (1, 5000, 28, 4), (3, 4099, 8, 1), (1, 9000, 6, 6), (3, 2500, 12, 3), (1, 700, 2, 1)])
def test_few_pairs_every_row_block_once(lib, monkeypatch, B, S, H, Hkv, pattern, arg0, arg1, waves):
    """Pairs that do not come out even over the XCDs: their row blocks are split."""
    dealing = Dealing(lib, monkeypatch, waves, LLM, pattern, B, S, H, Hkv, arg0, arg1)
    dealing.check()
    pairs = B * Hkv * dealing.plan.n_sets
    assert pairs % 8 != 0
    if pairs <= 4 and S > 1000:  # half of the XCDs or more would have nothing to do
        assert dealing.route()[0] * pairs >= 8


def test_plan_names_the_half_size_workgroups_for_image_gather0(lib):
    plan = _lib.IntraPlan()
    assert lib.intra_plan(IMAGE, GATHER0, 1, 16896, 24, 24, 128, 512, plan) == 0
    assert plan.waves == 4 and plan.pos_per_block == 128 and plan.lds_bytes < 80 * 1024
    assert lib.intra_plan(IMAGE, SCATTER, 1, 16896, 24, 24, 128, 512, plan) == 0
    assert plan.waves == 8 and plan.pos_per_block == 256
