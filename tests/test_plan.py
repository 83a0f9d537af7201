"""Host planner of the window kernel (C++ in libvdnh3.so) against the oracle's key sets.

Runs on the CPU: the planner is host code. Every query row must be covered by exactly
one work item, and the union of that item's valid key ranges must equal the oracle's
allowed set, with no key counted twice.
"""

from __future__ import annotations

import pytest
import torch

from oracle import window_oracle as wo


def _check_plan(built_lib, seq, vs, ve, frames, per_frame, bounds, anchors):
    from vdn_h3_amd import window

    bm, bn = built_lib.vdnh3_window_block_m(), built_lib.vdnh3_window_block_n()
    items, tiles, pairs = window.build_plan_host(seq, vs, ve, frames, per_frame, bounds, anchors)
    counts = items[:, 3].tolist()
    assert counts == sorted(counts, reverse=True), "items are longest-first"
    covered = torch.zeros(seq, dtype=torch.int64)
    for q0, q1, off, cnt in items.tolist():
        assert 0 <= q0 < q1 <= seq and q1 - q0 <= bm
        covered[q0:q1] += 1
        keys = []
        for ks, packed in tiles[off:off + cnt].tolist():
            lo, hi = packed & 0xFFFF, packed >> 16
            assert ks % bn == 0 and 0 <= lo < hi <= bn
            keys.extend(range(ks + lo, ks + hi))
        assert len(keys) == len(set(keys)), "a key tile range is repeated"
        assert max(keys) < seq
        for row in {q0, (q0 + q1) // 2, q1 - 1}:
            want = set()
            for a, b in wo.row_key_intervals(row, seq, vs, ve, frames, per_frame, bounds, anchors):
                want |= set(range(a, b))
            assert set(keys) == want, (row, anchors)
    assert bool((covered == 1).all())
    assert pairs == wo.pair_count(seq, vs, ve, frames, per_frame, bounds, anchors)


@pytest.mark.parametrize("anchors", wo.ANCHOR_FRAME_MODES)
@pytest.mark.parametrize("chunk,radius", [(0, 0), (0, 2), (3, 1), (4, 2), (5, 1)])
def test_plan_small_geometries(built_lib, anchors, chunk, radius):
    frames, per_frame, vs, after = 11, 3, 4, 2
    ve = vs + frames * per_frame
    _check_plan(built_lib, ve + after, vs, ve, frames, per_frame, wo.window_bounds(frames, radius, chunk), anchors)


@pytest.mark.parametrize("frames,per_frame,text", [(7, 64, 16), (13, 64, 16), (31, 1296, 512), (12, 100, 0)])
def test_plan_packed_layouts(built_lib, frames, per_frame, text):
    bounds = wo.window_bounds(frames, 1, 5)
    _check_plan(built_lib, text + frames * per_frame, text, text + frames * per_frame, frames, per_frame, bounds,
                "both")


def test_plan_validation_errors(built_lib):
    from vdn_h3_amd import window

    with pytest.raises(ValueError, match="does not contain its query frame"):
        window.build_plan_host(40, 4, 34, 3, 10, [(0, 2), (0, 2), (0, 0)], "none")
    with pytest.raises(ValueError, match="one entry per frame"):
        window.build_plan_host(40, 4, 34, 3, 10, [(0, 2)] * 2, "none")
    with pytest.raises(ValueError, match="must be positive"):
        window.build_plan_host(40, 4, 4, 0, 10, [], "none")
    with pytest.raises(ValueError, match="video range does not equal"):
        window.build_plan_host(40, 4, 33, 3, 10, window.window_bounds(3, 1), "none")
    with pytest.raises(ValueError, match="anchor_frames"):
        window.build_plan_host(40, 4, 34, 3, 10, window.window_bounds(3, 1), "sideways")


@pytest.mark.parametrize("heads", [1, 2, 7, 40])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("text,frames,per_frame", [(16, 13, 64), (1, 1, 1), (300, 20, 320), (512, 1, 1296), (512, 31, 1296)])
def test_item_height_and_key_splits_rule(built_lib, heads, dim, text, frames, per_frame):
    """The rule keeps to the kernel's limits, and a call that fills the 256 CUs several times over is left whole."""
    from vdn_h3_amd import window

    seq = text + frames * per_frame
    geometry = (seq, text, seq, frames, per_frame, wo.window_bounds(frames, 1, 5), "both")
    plan = window.make_plan(*geometry, torch.device("cpu"), heads, dim)
    counts, rows = plan.items[:, 3], plan.items[:, 1] - plan.items[:, 0]
    assert plan.block_m in (64, 128, 256) and int(rows.max()) <= plan.block_m and int(rows.sum()) == seq
    assert 1 <= plan.splits <= int(counts.min())
    if -(-seq // 256) * heads >= 1024:
        assert (plan.block_m, plan.splits) == (256, 1)
    whole = window.make_plan(*geometry, torch.device("cpu"))
    assert (whole.block_m, whole.splits, whole.pairs_per_head) == (256, 1, plan.pairs_per_head)


@pytest.mark.parametrize("hold", [list, tuple, torch.tensor, lambda b: torch.tensor(b).numpy(),
                                  lambda b: [torch.tensor(p) for p in b]])
def test_cached_plan_whatever_holds_the_bounds(built_lib, hold):
    from vdn_h3_amd import window

    bounds = wo.window_bounds(5, 1, 2)
    cache, device = window.WindowAttentionCache(), torch.device("cpu")
    geometry = lambda b: (516, 16, 516, 5, 100, b, "both", device, 2, 64)  # noqa: E731
    first = cache.plan(*geometry(bounds))
    assert cache.plan(*geometry(hold(bounds))) is first
    assert cache.plan(*geometry(hold(bounds))) is first and len(cache) == 1
    for wrong in ([(0, 1, 2), (3,)], [(0,)] * 5, []):
        with pytest.raises(ValueError):
            cache.plan(*geometry(wrong))


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("seq,heads", [(6700, 1), (8364, 1), (10598, 2), (16441, 3), (23883, 2), (23883, 5), (40688, 1),
                                       (40688, 3), (40688, 5)])
def test_key_splits_save_rounds(built_lib, seq, heads, dim):
    """Items of one length: an XCD's 32 CUs take its eighth of the items' splits in rounds, and a choice with splits takes
    less in those rounds than whole items do (33 workgroups on an XCD are two rounds)."""
    from vdn_h3_amd import window

    def rounds(block_m, splits):
        per_xcd = -(-(-(-seq // block_m) * heads) // 8)
        return -(-per_xcd * splits // 32) * (-(-seq // 96) / splits + 5)

    plan = window.make_plan(seq, 0, seq, 1, seq, [(0, 0)], "none", torch.device("cpu"), heads, dim)
    assert (plan.block_m, plan.splits) == (256, 1) or rounds(plan.block_m, plan.splits) < rounds(256, 1)
