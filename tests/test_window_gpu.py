"""Parity of the HIP window-attention kernel with the CPU oracle (GPU).

Tolerance (bf16 in / bf16 out, fp32 softmax): max |got - want| <= 2e-2 and cosine >= 0.9995
against the fp32 oracle on the same bf16 inputs; the reference's own backend parity gate
(``vdn_h3/autotune.py:133``, ``allclose(atol=2e-2, rtol=4e-2)``) is checked as well.
"""

from __future__ import annotations

import pytest
import torch

from oracle import window_oracle as wo

pytestmark = pytest.mark.gpu

ATOL = 2e-2
MIN_COS = 0.9995


def assert_parity(got, want, atol=ATOL, min_cos=MIN_COS):
    got = got.float().cpu()
    want = want.float().cpu()
    assert got.shape == want.shape
    assert torch.isfinite(got).all()
    err = (got - want).abs().max().item()
    cos = torch.nn.functional.cosine_similarity(got.double().flatten(), want.double().flatten(), dim=0).item()
    assert err <= atol and cos >= min_cos, f"max abs {err:.3e}, cosine {cos:.6f}"
    assert torch.allclose(got, want, atol=2e-2, rtol=4e-2)


def _run(device, seq, vs, ve, frames, per_frame, heads, dim, bounds, anchors, seed, strided=True, gate=None):
    from vdn_h3_amd import window

    gen = torch.Generator().manual_seed(seed)
    qkv = torch.randn(seq, 3 * heads * dim, generator=gen).to(torch.bfloat16)
    q, k, v = [t.view(seq, heads, dim) for t in qkv.split(heads * dim, dim=-1)]
    dq = qkv.to(device)
    gq, gk, gv = [t.view(seq, heads, dim) for t in dq.split(heads * dim, dim=-1)]
    if not strided:
        gq, gk, gv = gq.contiguous(), gk.contiguous(), gv.contiguous()
    scale = dim ** -0.5
    out = window.window_softmax_hip(gq, gk, gv, vs, ve, frames, per_frame, bounds, scale, anchors,
                                    gate=None if gate is None else gate.to(device))
    torch.cuda.synchronize()
    want = wo.window_attention_grouped(q, k, v, vs, ve, frames, per_frame, bounds, scale, anchors)
    if gate is not None:
        want = (want.to(torch.bfloat16) * gate.reshape(seq, heads, 1)).float()
    return out, want


@pytest.mark.parametrize("anchors", wo.ANCHOR_FRAME_MODES)
@pytest.mark.parametrize("chunk,radius", [(0, 2), (3, 1), (4, 2)])
def test_small_geometry_all_anchor_modes(device, anchors, chunk, radius):
    # the reference's window test geometry (11 frames x 3 tokens, 4 rows before, 2 after), head_dim 64
    frames, per_frame, vs = 11, 3, 4
    ve = vs + frames * per_frame
    seq = ve + 2
    bounds = wo.window_bounds(frames, radius, chunk)
    print(f"case small anchors={anchors} chunk={chunk} radius={radius}", flush=True)
    out, want = _run(device, seq, vs, ve, frames, per_frame, 2, 64, bounds, anchors, 1000 + 10 * chunk + radius)
    assert_parity(out, want)


@pytest.mark.parametrize("frames", [7, 13])
@pytest.mark.parametrize("dim", [64, 128])
def test_packed_layout_8x8_frames(device, frames, dim):
    # 16 text rows + frames x 64 tokens; 7 frames is full cover (dense), 13 frames is windowed
    per_frame, text, heads = 64, 16, 2
    seq = text + frames * per_frame
    bounds = wo.window_bounds(frames, 1, 5)
    print(f"case packed frames={frames} dim={dim}", flush=True)
    out, want = _run(device, seq, text, seq, frames, per_frame, heads, dim, bounds, "both", 7 + frames)
    assert_parity(out, want)


def test_ragged_tiles_and_contiguous_operands(device):
    # frames of 100 tokens: neither query blocks (128) nor key tiles (64) align with frames
    frames, per_frame, text, heads, dim = 12, 100, 40, 3, 128
    seq = text + frames * per_frame + 24
    bounds = wo.window_bounds(frames, 1, 3)
    print("case ragged", flush=True)
    for strided in (True, False):
        out, want = _run(device, seq, text, text + frames * per_frame, frames, per_frame, heads, dim, bounds,
                         "columns", 99, strided=strided)
        assert_parity(out, want)


def test_fused_gate(device):
    frames, per_frame, text, heads, dim = 13, 64, 16, 2, 128
    seq = text + frames * per_frame
    gate = torch.sigmoid(torch.randn(seq, heads, generator=torch.Generator().manual_seed(5))).to(torch.bfloat16)
    print("case gate", flush=True)
    out, want = _run(device, seq, text, seq, frames, per_frame, heads, dim, wo.window_bounds(frames, 1, 5), "both",
                     31, gate=gate)
    assert_parity(out, want)


@pytest.mark.parametrize("input_scale", [1.0, 128 ** -0.5])
def test_full_shape_sampled_rows(device, input_scale):
    """40 688 tokens x 40 heads x 128: the whole problem on the GPU, exact oracle on one row of every work
    item of the plan (at a position that walks through the item) plus the layout's boundary rows, all 40
    heads. Inputs ~ N(0, 1) (a sharp softmax) and ~ N(0, 1) / sqrt(128) (the benchmark's inputs)."""
    from vdn_h3_amd import synth, window

    w = synth.WINDOW_FULL
    print(f"case full shape S={w.layout.seq_len} input scale {input_scale:.4f}", flush=True)
    qkv, q, k, v, lay, _ = synth.window_inputs(w, device=device, input_scale=input_scale)
    out = window.window_softmax_hip(q, k, v, lay.video_start, lay.video_end, lay.num_frames, lay.tokens_per_frame,
                                    lay.bounds, w.scale, lay.anchor_frames)
    torch.cuda.synchronize()
    items, _, _ = window.build_plan_host(lay.seq_len, lay.video_start, lay.video_end, lay.num_frames,
                                         lay.tokens_per_frame, lay.bounds, lay.anchor_frames)
    host = qkv.cpu()
    hq, hk, hv = synth.split_qkv(host, w.heads, w.head_dim)
    T, vs = lay.tokens_per_frame, lay.video_start
    rows = {0, 511, vs, vs + T - 1, vs + T, vs + 2 * T + 127, vs + 2 * T + 128, vs + 5 * T - 1, vs + 5 * T,
            vs + 12 * T + 700, vs + 25 * T, vs + 29 * T + 1295, vs + 30 * T, lay.seq_len - 1}
    for i, (q0, q1, _, _) in enumerate(items.tolist()):
        rows.add(q0 + (37 * i) % (q1 - q0))
    rows = sorted(rows)
    print(f"  {len(rows)} rows ({items.shape[0]} work items)", flush=True)
    want = wo.window_attention_rows(hq, hk, hv, rows, lay.video_start, lay.video_end, lay.num_frames, T, lay.bounds,
                                    w.scale, lay.anchor_frames)
    assert_parity(out.cpu()[rows], want)


@pytest.mark.parametrize("dim", [32, 80, 96])
def test_head_dims_below_128_run_with_zero_channels(device, dim):
    """Head dims other than 64 / 128 (the reference's window op is shape-generic, vdn_h3/window.py:277-313) run
    at the next kernel head dim with zero channels added; the scale stays the caller's D^-1/2. The bar is the
    kernel's own (max-abs 2e-2, cosine 0.9995 against the fp32 oracle at the true head dim), with the gate, and
    into a caller's output."""
    from vdn_h3_amd import window

    frames, per_frame, vs, heads = 7, 24, 10, 3
    ve = vs + frames * per_frame
    seq = ve + 6
    bounds = wo.window_bounds(frames, 1, 3)
    print(f"case window head_dim={dim}", flush=True)
    gate = torch.sigmoid(torch.randn(seq, heads, generator=torch.Generator().manual_seed(5))).to(torch.bfloat16)
    got, want = _run(device, seq, vs, ve, frames, per_frame, heads, dim, bounds, "both", seed=dim, gate=gate)
    assert got.shape == (seq, heads, dim)
    assert_parity(got, want)
    gen = torch.Generator().manual_seed(dim + 1)
    q, k, v = [torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16).to(device) for _ in range(3)]
    out = torch.empty(seq, heads, dim, dtype=torch.bfloat16, device=device)
    res = window.window_softmax_hip(q, k, v, vs, ve, frames, per_frame, bounds, dim ** -0.5, "both", out=out)
    torch.cuda.synchronize()
    assert res is out
    assert_parity(out, wo.window_attention_grouped(q.cpu(), k.cpu(), v.cpu(), vs, ve, frames, per_frame, bounds,
                                                   dim ** -0.5, "both"))
    with pytest.raises(ValueError, match="head dims 1 to 128"):
        big = torch.zeros(seq, 1, 160, dtype=torch.bfloat16, device=device)
        window.window_softmax_hip(big, big, big, vs, ve, frames, per_frame, bounds, 160 ** -0.5, "both")


def test_calls_hold_no_memory_beyond_their_output(device):
    """The op keeps nothing between calls but the cached tile plan (the reference releases its per-group buffers,
    ``tests/test_window.py:14-38``): after a warm call, further calls whose outputs are dropped leave the
    allocated device memory where it was, and a kept output adds exactly its own size."""
    from vdn_h3_amd import window

    frames, per_frame, text, heads, dim = 13, 64, 16, 2, 128
    seq = text + frames * per_frame
    print("case window memory", flush=True)
    qkv = torch.randn(seq, 3 * heads * dim, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(device)
    q, k, v = [t.view(seq, heads, dim) for t in qkv.split(heads * dim, dim=-1)]
    cache = window.WindowAttentionCache(limit=4)
    args = (text, seq, frames, per_frame, wo.window_bounds(frames, 1, 5), dim ** -0.5, "both", cache)
    first = window.window_softmax_hip(q, k, v, *args)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated(device)
    for _ in range(3):
        window.window_softmax_hip(q, k, v, *args)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated(device) == base
    kept = window.window_softmax_hip(q, k, v, *args)
    torch.cuda.synchronize()
    grown = torch.cuda.memory_allocated(device) - base
    assert grown == kept.untyped_storage().nbytes() or grown == -(-kept.untyped_storage().nbytes() // 512) * 512
    assert torch.equal(kept, first)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("block_m,splits", [(256, 2), (256, 3), (128, 1), (128, 5), (64, 1), (64, 4), (256, "all")])
def test_key_splits_and_short_items(device, dim, block_m, splits):
    """Every item height and any number of key splits, up to one tile each, against the oracle, with and without a gate."""
    from vdn_h3_amd import window

    frames, per_frame, text, heads = 9, 61, 37, 3  # ragged: items of 37, 61 and 305 rows, masked tile edges
    seq = text + frames * per_frame
    bounds = wo.window_bounds(frames, 1, 4)
    print(f"case splits D={dim} block_m={block_m} splits={splits}", flush=True)
    geometry = (seq, text, seq, frames, per_frame, bounds, "both")
    items, tiles, pairs = window.build_plan_host(*geometry, block_m)
    fewest = int(items[:, 3].min())
    assert int((items[:, 1] - items[:, 0]).max()) <= block_m and fewest >= 5
    plan = window.WindowPlan(items.to(device), tiles.to(device), items.shape[0], tiles.shape[0], pairs, block_m,
                             fewest if splits == "all" else splits)
    gen = torch.Generator().manual_seed(17)
    q, k, v = (torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16) for _ in range(3))
    gate = torch.sigmoid(torch.randn(seq, heads, generator=gen)).to(torch.bfloat16)
    want = wo.window_attention_grouped(q, k, v, *geometry[1:6], dim ** -0.5, "both")
    args = (q.to(device), k.to(device), v.to(device), *geometry[1:6], dim ** -0.5, "both")
    out = window.window_softmax_hip(*args, plan=plan)
    gated = window.window_softmax_hip(*args, plan=plan, gate=gate.to(device))
    torch.cuda.synchronize()
    assert_parity(out, want)
    assert torch.equal(gated, out * gate.to(device)[..., None])


@pytest.mark.parametrize("dim", [64, 128])
def test_values_sum_sixteen_keys_at_a_time(device, dim):
    """The PV product adds the keys of one aligned group of 16 before those of the next: large values that cancel within
    a group leave no rounding behind for a small one in the next group."""
    from vdn_h3_amd import window

    seq, heads = 192, 2
    q = torch.zeros(seq, heads, dim, dtype=torch.bfloat16, device=device)  # equal scores: every probability is 1
    v = torch.zeros_like(q)
    for group in range(seq // 32):  # a channel per pair of groups
        v[32 * group + 4, :, group], v[32 * group + 8, :, group], v[32 * group + 16, :, group] = 2.0 ** 30, -2.0 ** 30, 1
    out = window.window_softmax_hip(q, q, v, 0, seq, 1, seq, [(0, 0)], dim ** -0.5, "none",
                                    plan=window.dense_plan(seq, device))
    want = torch.zeros_like(out)
    want[..., :seq // 32] = 1 / seq
    assert torch.equal(out, want)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("value", [float("-inf"), torch.finfo(torch.bfloat16).min, -1e9])
@pytest.mark.parametrize("block_m,splits", [(256, 1), (256, 3), (64, 4), (256, "all")])
def test_masked_tiles_add_nothing(device, dim, value, block_m, splits):
    """Keys masked through a channel of q and k, whole key tiles of them: at the front of an item's or of a split's tiles
    too, they take no part, and a row with no other key is NaN."""
    from vdn_h3_amd import window

    frames, per_frame, text, heads = 9, 192, 192, 2  # 96-key tiles: two to a frame
    seq = text + frames * per_frame
    geometry = (seq, text, seq, frames, per_frame, wo.window_bounds(frames, 1), "both")
    items, tiles, pairs = window.build_plan_host(*geometry, block_m)
    fewest = int(items[:, 3].min())
    plan = window.WindowPlan(items.to(device), tiles.to(device), items.shape[0], tiles.shape[0], pairs, block_m,
                             fewest if splits == "all" else splits)
    gen = torch.Generator().manual_seed(19)
    q, k, v = (torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16) for _ in range(3))
    q[..., -1], k[..., -1] = 1, 0
    k[:96, :, -1] = value   # the first tile of every item
    for frame in (2, 4):    # the first tiles of a split, in three splits of the rows of frames 0 (20 tiles) and 5 (12)
        k[text + frame * 192:text + (frame + 1) * 192, :, -1] = value
    k[-96:, 1, -1] = value  # the last tile, of one head
    want = wo.window_attention_grouped(q, k, v, *geometry[1:6], dim ** -0.5, "both")
    assert bool(want.isfinite().all())
    args = (*geometry[1:6], dim ** -0.5, "both")
    out = window.window_softmax_hip(q.to(device), k.to(device), v.to(device), *args, plan=plan)
    assert_parity(out, want)
    if value == float("-inf"):
        k[..., -1] = value
        out = window.window_softmax_hip(q.to(device), k.to(device), v.to(device), *args, plan=plan)
        assert bool(out.isnan().all())


@pytest.mark.parametrize("dim", [64, 128])
def test_more_splits_than_tiles(device, dim):
    """The splits past an item's tile count read no tile and add nothing; items of the same plan differ in count."""
    from vdn_h3_amd import window

    frames, per_frame, text, heads = 9, 61, 37, 3
    seq = text + frames * per_frame
    geometry = (seq, text, seq, frames, per_frame, wo.window_bounds(frames, 1), "columns")
    items, tiles, pairs = window.build_plan_host(*geometry, 64)
    counts = items[:, 3]
    assert int(counts.min()) < int(counts.max()) < 64
    gen = torch.Generator().manual_seed(29)
    q, k, v = (torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16) for _ in range(3))
    want = wo.window_attention_grouped(q, k, v, *geometry[1:6], dim ** -0.5, "columns")
    for splits in (int(counts.min()) + 1, 64):
        print(f"case splits past the tiles D={dim} splits={splits}", flush=True)
        plan = window.WindowPlan(items.to(device), tiles.to(device), items.shape[0], tiles.shape[0], pairs, 64, splits)
        out = window.window_softmax_hip(q.to(device), k.to(device), v.to(device), *geometry[1:6], dim ** -0.5, "columns",
                                        plan=plan)
        assert_parity(out, want)


@pytest.mark.parametrize("normed", [False, True])
def test_items_stay_whole_without_memory_for_partials(device, monkeypatch, normed):
    """A call whose partial results find no memory runs its items whole: the result of the same plan without splits."""
    from dataclasses import replace

    from vdn_h3_amd import _lib, window

    seq, heads, dim = 700, 2, 128
    plan = replace(window.dense_plan(seq, device), splits=3)
    size = _lib.lib().vdnh3_window_partial_bytes(seq, heads, dim, 3)
    gen = torch.Generator().manual_seed(31)
    q, k, v = (torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16).to(device) for _ in range(3))
    weight = torch.ones(dim, dtype=torch.bfloat16, device=device)

    def call(plan):
        geometry = (0, seq, 1, seq, [(0, 0)])
        if normed:
            return window.window_softmax_normed(q, k, v, weight, weight, 1e-6, 1e-6, *geometry, dim ** -0.5, "none",
                                                plan=plan)
        return window.window_softmax_hip(q, k, v, *geometry, dim ** -0.5, "none", plan=plan)

    whole, split, empty = call(replace(plan, splits=1)), call(plan), torch.empty
    refused = []

    def full(*shape, **options):
        if shape[0] == size:
            refused.append(size)
            raise torch.OutOfMemoryError("out of memory")
        return empty(*shape, **options)

    monkeypatch.setattr(torch, "empty", full)
    out = call(plan)
    assert refused and torch.equal(out, whole) and not torch.equal(split, whole)


def test_whole_items_keep_a_heads_bits_in_any_company(device):
    """With a plan made without the number of heads a head computed alone has the bits it has among others."""
    from vdn_h3_amd import window

    frames, per_frame, text, heads, dim = 13, 300, 100, 6, 128
    seq = text + frames * per_frame
    geometry = (text, seq, frames, per_frame, wo.window_bounds(frames, 1, 5))
    gen = torch.Generator().manual_seed(37)
    q, k, v = (torch.randn(seq, heads, dim, generator=gen).to(torch.bfloat16).to(device) for _ in range(3))
    plan = window.make_plan(seq, *geometry, "both", device)
    assert plan.splits == 1 and window.make_plan(seq, *geometry, "both", device, 1, dim).splits > 1
    args = (*geometry, dim ** -0.5, "both")
    together = window.window_softmax_hip(q, k, v, *args, plan=plan)
    for head in (0, heads - 1):
        alone = window.window_softmax_hip(*(t[:, head:head + 1] for t in (q, k, v)), *args, plan=plan)
        assert torch.equal(alone, together[:, head:head + 1])
