"""Float32 attention that finishes the q/k/v product itself: the bits of the kernels one after the other."""

import math

import pytest
import torch

from test_kernels_gpu import paged_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops

    ops.load()
    return ops


@pytest.mark.parametrize("units", [4096, 8])  # short items and a merge; whole requests, of which some have more blocks than a workgroup has waves
@pytest.mark.parametrize("heads, kv, hd, page, window, n_parts, extras", [
    (14, 2, 64, 16, None, 3, "bias table"),
    (28, 4, 128, 16, None, 8, "bias table"),
    (12, 4, 128, 8, None, 11, "table"),      # more slices than the kernel reads at once
    (20, 1, 32, 4, None, 1, ""),             # more heads a kv head than rows of a tile: two workgroups a kv head, one of them writes; nothing turned
    (6, 3, 96, 24, None, 2, "bias table"),   # head and page size no powers of two
    (8, 8, 16, 16, None, 5, "table"),
    (6, 2, 80, 16, 37, 7, "bias table slopes scale"),
])
def test_the_same_bits(ops, units, heads, kv, hd, page, window, n_parts, extras):
    from from_scratch_inference_engine_amd.parts.attention import AttentionPlanner

    pasts = [0, 19, 15, 16, 31, 600, 127, 128, 1500, 1023, 7, 255]
    t, width = len(pasts), (heads + 2 * kv) * hd
    AttentionPlanner.compute_units = units
    try:
        case = paged_case([(p, 1) for p in pasts], heads, kv, hd, page, torch.float32, seed=heads + hd, window=window)
    finally:
        AttentionPlanner.compute_units = None
    plan = case["plan"]
    assert not plan["mfma"] and plan["single"] and not plan["n_large"]
    g = torch.Generator().manual_seed(5)
    parts = torch.randn(n_parts, t, width, generator=g).cuda()
    bias = torch.randn(width, generator=g).cuda() if "bias" in extras else None
    positions = torch.tensor(pasts, dtype=torch.int32).cuda()
    inv_freq = torch.pow(torch.tensor(1e4, dtype=torch.float64), -torch.arange(0, hd, 2, dtype=torch.float64) / hd).cuda()
    table = ops.rope_table(positions, inv_freq) if "table" in extras else None
    more = {}
    if "slopes" in extras:
        more = {"slopes": torch.rand(heads, generator=g).cuda() * 0.1, "row_scale": torch.rand(t, generator=g).cuda() + 0.5}
    tables = case["tables"]
    slots = torch.tensor([int(tables[s, p // page]) * page + p % page for s, p in enumerate(pasts)], dtype=torch.int32).cuda()
    slots[3] = -1  # (a token that goes nowhere is attended to all the same)
    items, merges, bt = torch.from_numpy(plan["items"]).cuda(), torch.from_numpy(plan["merges"]).cuda(), tables.cuda()
    scale = 1.0 / math.sqrt(hd)
    outs, pools = [], []
    for joined in (False, True):
        k, v = case["k_pool"].cuda().clone(), case["v_pool"].cuda().clone()
        out = torch.zeros(t, heads * hd).cuda()
        partials = torch.zeros(max(plan["n_partial"], 1) * heads * (hd + 2)).cuda()
        if joined:
            assert ops.attention_f32_qkv_ok(hd, page)
            ops.attention_mfma_qkv(parts, bias, table, slots, k, v, bt, items, plan["n_small"], out, partials, heads, kv, hd, window, scale, **more)
        else:
            qkv = torch.empty(t, width).cuda()
            ops.rope_kv_write(qkv, positions, heads, kv, hd, None, slots=slots, k_pool=k, v_pool=v, page_size=page, bias=bias, cos_sin=table,
                              parts=parts, by_rows=True)
            ops.attention_scalar(qkv, width, k, v, bt, items, plan["n_small"], out, partials, heads, kv, hd, window, scale, t, **more)
        if plan["n_merges"]:
            ops.attention_merge(partials, merges, plan["n_merges"], out, heads, hd)
        outs.append(out), pools.append((k, v))
    assert torch.equal(pools[0][0], pools[1][0]) and torch.equal(pools[0][1], pools[1][1])
    rows = [r for r in range(t) if r != 3]  # (one after the other the token without a slot is read from where it was not written)
    assert torch.equal(outs[0][rows], outs[1][rows]) and outs[0].abs().max() > 0.1


def test_refusals(ops):
    def call(hd, page):
        return ops.attention_mfma_qkv(torch.zeros(1, 1, 3 * hd).cuda(), None, None, torch.zeros(1, dtype=torch.int32).cuda(), torch.zeros(2, 1, page, hd).cuda(),
                                      torch.zeros(2, 1, hd, page).cuda(), torch.zeros(1, 1, dtype=torch.int32).cuda(), torch.zeros(1, 8, dtype=torch.int32).cuda(), 1,
                                      torch.zeros(1, hd).cuda(), None, 1, 1, hd, None, 1.0)

    for hd, page in ((144, 16), (40, 16), (64, 6)):
        assert not ops.attention_f32_qkv_ok(hd, page)
        with pytest.raises(ops.KernelError):
            call(hd, page)
    with pytest.raises(ops.KernelError, match="k_pool|out"):  # all of one type
        ops.attention_mfma_qkv(torch.zeros(1, 1, 192).cuda(), None, None, torch.zeros(1, dtype=torch.int32).cuda(), torch.zeros(2, 1, 16, 64).cuda(),
                               torch.zeros(2, 1, 64, 16).cuda(), torch.zeros(1, 1, dtype=torch.int32).cuda(), torch.zeros(1, 8, dtype=torch.int32).cuda(), 1,
                               torch.zeros(1, 64, dtype=torch.bfloat16).cuda(), None, 1, 1, 64, None, 1.0)


@pytest.mark.parametrize("heads, kv, hd, page, n_parts, table", [
    (14, 2, 64, 16, 7, True), (16, 1, 128, 8, 3, True), (32, 2, 96, 16, 9, True),  # (sixteen heads of 96 and 128: more columns than four waves have threads)
    (3, 3, 16, 4, 1, False), (20, 1, 64, 16, 2, False)])
def test_short_items_give_the_same_bits_on_four_waves(ops, heads, kv, hd, page, n_parts, table):
    short_items_on_four_waves(ops, heads, kv, hd, page, n_parts, table, [0, 5, 15, 16, 63, 64, 200, 330], None)


@pytest.mark.parametrize("window", [200, 263, 320])
def test_short_items_of_a_window_give_the_same_bits_on_four_waves(ops, window):
    short_items_on_four_waves(ops, 14, 2, 64, 16, 7, True, [0, 199, 206, 330, 471, 600, 601, 1000], window)


def short_items_on_four_waves(ops, heads, kv, hd, page, n_parts, table, pasts, window):
    from from_scratch_inference_engine_amd.parts.attention import AttentionPlanner

    t, width = len(pasts), (heads + 2 * kv) * hd
    AttentionPlanner.compute_units = 4096  # (items of 64 keys)
    try:
        case = paged_case([(p, 1) for p in pasts], heads, kv, hd, page, torch.float32, seed=heads, window=window)
    finally:
        AttentionPlanner.compute_units = None
    plan = case["plan"]
    assert plan["short_items"] and plan["n_partial"] and all(it[5] - it[4] <= 64 for it in plan["items"][:plan["n_small"]])
    g = torch.Generator().manual_seed(9)
    parts, bias = torch.randn(n_parts, t, width, generator=g).cuda(), torch.randn(width, generator=g).cuda()
    angles = torch.randn(t, hd, generator=g).cuda() if table else None
    tables = case["tables"]
    slots = torch.tensor([int(tables[s, p // page]) * page + p % page for s, p in enumerate(pasts)], dtype=torch.int32).cuda()
    items, bt = torch.from_numpy(plan["items"]).cuda(), tables.cuda()
    got = []
    for short in (False, True):
        k, v = case["k_pool"].cuda().clone(), case["v_pool"].cuda().clone()
        out, partials = torch.zeros(t, heads * hd).cuda(), torch.zeros(plan["n_partial"] * heads * (hd + 2)).cuda()
        ops.attention_mfma_qkv(parts, bias, angles, slots, k, v, bt, items, plan["n_small"], out, partials, heads, kv, hd, window, hd ** -0.5, short_items=short)
        got.append((out, partials, k, v))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and got[0][1].abs().max() > 0.1
