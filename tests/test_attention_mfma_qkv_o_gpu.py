"""The output projection in attention's own launch: the heads of the two launches, times the weight in float32."""

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


@pytest.mark.parametrize("rows", [2, 3, 4])
@pytest.mark.parametrize("heads, kv, hd, n, page, window, n_parts, extras", [
    (14, 2, 64, 896, 16, None, 3, "bias table"),
    (12, 2, 128, 1536, 16, None, 2, "bias table"),
    (32, 2, 128, 37, 8, None, 9, "table"),  # sixteen heads a kv head: four loads a row; rows that are no multiple of a workgroup's
    (3, 3, 64, 16, 16, 37, 1, ""),          # one head, less than a wave's load
    (1, 1, 128, 1, 24, None, 5, "table"),
])
def test_sums(ops, rows, heads, kv, hd, n, page, window, n_parts, extras):
    from from_scratch_inference_engine_amd.parts.attention import AttentionPlanner

    pasts = [0, 60, 31, 32, 127, 15, 333]  # (the last has more blocks of keys than the variant has waves)
    t, width = len(pasts), (heads + 2 * kv) * hd
    AttentionPlanner.compute_units = 1
    try:
        case = paged_case([(p, 1) for p in pasts], heads, kv, hd, page, torch.bfloat16, seed=heads + n, window=window)
    finally:
        AttentionPlanner.compute_units = None
    plan = case["plan"]
    assert plan["mfma"] and plan["single"] and not plan["n_large"] and not plan["n_partial"]
    g = torch.Generator().manual_seed(6)
    parts = torch.randn(n_parts, t, width, generator=g).cuda()
    bias = torch.randn(width, generator=g).cuda() if "bias" in extras else None
    weight = torch.randn(n, heads * hd, generator=g).to(torch.bfloat16).cuda()
    positions = torch.tensor(pasts, dtype=torch.int32).cuda()
    inv_freq = torch.pow(torch.tensor(1e4, dtype=torch.float64), -torch.arange(0, hd, 2, dtype=torch.float64) / hd).cuda()
    table = ops.rope_table(positions, inv_freq) if "table" in extras else None
    tables = case["tables"]
    slots = torch.tensor([int(tables[s, p // page]) * page + p % page for s, p in enumerate(pasts)], dtype=torch.int32).cuda()
    slots[3] = -1
    items, bt = torch.from_numpy(plan["items"]).cuda(), tables.cuda()
    k, v = case["k_pool"].cuda().clone(), case["v_pool"].cuda().clone()
    kj, vj = k.clone(), v.clone()
    out = torch.zeros(t, heads * hd, dtype=torch.bfloat16).cuda()
    ops.attention_mfma_qkv(parts, bias, table, slots, k, v, bt, items, plan["n_small"], out, None, heads, kv, hd, window, 1 / math.sqrt(hd))
    sums = torch.full((kv, t, n), float("nan")).cuda()
    ops.attention_mfma_qkv(parts, bias, table, slots, kj, vj, bt, items, plan["n_small"], sums, None, heads, kv, hd, window, 1 / math.sqrt(hd),
                           o_weight=weight, o_rows=rows)
    assert torch.equal(k, kj) and torch.equal(v, vj)
    # (the heads are the same kernel's, so the same bits; what is left is a float32 sum of heads / kv * head_dim products)
    x = out.double().view(t, kv, -1).transpose(0, 1).contiguous()
    w = weight.double().view(n, kv, -1).permute(1, 2, 0).contiguous()
    bound = torch.bmm(x.abs(), w.abs()) * (heads // kv * hd) * 2.0 ** -24 + 1e-30
    assert ((sums.double() - torch.bmm(x, w)).abs() <= bound).all()


def test_rule(ops):
    units, rows = ops.compute_units(), ops.attention_mfma_qkv_o_rows
    assert rows(1, 14, 2, 64, 16, 896) == 2 and rows(2, 14, 2, 64, 16, 896) == 3 and rows(1, 12, 2, 128, 16, 1536) == 3
    assert rows(1, 16, 16, 128, 16, 2048) == 0 and rows(units, 14, 2, 64, 16, 896) == 0  # more workgroups than units
    assert rows(1, 16, 1, 128, 16, 2304) == 2 and rows(2, 16, 1, 128, 16, 2304) == 0  # 9 MB of weights, and 19
    assert rows(1, 34, 2, 64, 16, 896) == 0 and rows(1, 14, 2, 96, 16, 896) == 0 and rows(1, 14, 2, 64, 12, 896) == 0 and rows(0, 14, 2, 64, 16, 896) == 0


def test_refusals(ops):
    def call(**kw):
        a = dict(hd=64, page=16, heads=2, n=8, out=(1, 1, 8), o_rows=2, cols=None) | kw
        hd, page, heads = a["hd"], a["page"], a["heads"]
        ops.attention_mfma_qkv(torch.zeros(1, 1, (heads + 2) * hd).cuda(), None, None, torch.zeros(1, dtype=torch.int32).cuda(),
                               torch.zeros(2, 1, page, hd, dtype=torch.bfloat16).cuda(), torch.zeros(2, 1, hd, page, dtype=torch.bfloat16).cuda(),
                               torch.zeros(1, 1, dtype=torch.int32).cuda(), torch.zeros(1, 8, dtype=torch.int32).cuda(), 1,
                               torch.zeros(a["out"]).cuda(), None, heads, 1, hd, None, 1.0,
                               o_weight=torch.zeros(a["n"], a["cols"] or heads * hd, dtype=torch.bfloat16).cuda(), o_rows=a["o_rows"])

    for bad in (dict(hd=96), dict(heads=17), dict(o_rows=0), dict(o_rows=5), dict(out=(1, 1, 9)), dict(cols=64), dict(page=12)):
        with pytest.raises(ops.KernelError):
            call(**bad)
    call()  # (an item without queries)
