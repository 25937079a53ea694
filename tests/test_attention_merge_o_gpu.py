"""The output projection in the launch that merges a decode step's cut items: the heads of the merge alone, times the weight in float32."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops

    ops.load()
    return ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("heads, kv, hd, n, splits", [
    (14, 2, 64, 896, [3, 8]), (12, 2, 128, 1536, [1, 9]),
    (32, 2, 128, 37, [2, 0, 30]),          # sixteen heads a kv head, two a wave; a token that attention has left whole
    (3, 3, 64, 16, [32, 0]), (1, 1, 64, 1, [5]),
])
def test_sums(ops, dtype, rows, heads, kv, hd, n, splits):
    t, g = len(splits), torch.Generator().manual_seed(heads + n)
    slots = sum(splits)
    records = torch.randn(slots, heads, hd + 2, generator=g)
    records[..., hd + 1] = records[..., hd + 1].abs() + 0.5   # the denominators
    records[:, 0, hd] = -float("inf")                          # a head that has seen no key in any record: nothing, not NaN
    records[:, 0, :hd] = records[:, 0, hd + 1] = 0
    if max(splits) > 2:
        at = sum(splits[:splits.index(max(splits))])
        records[at + 1, -1, hd] = -float("inf")                # and one that has seen none in one of them
        records[at + 1, -1, :hd] = records[at + 1, -1, hd + 1] = 0
    order = list(range(t))[::-1]                                # (the rows in any order, their records one after the other)
    merges = torch.tensor([(r, sum(splits[:r]), splits[r], 1) for r in order], dtype=torch.int32).cuda()
    weight = torch.randn(n, heads * hd, generator=g).to(dtype).cuda()
    whole = torch.randn(t, heads * hd, generator=g).to(dtype).cuda()
    partials = records.reshape(-1).cuda()
    merged = whole.clone()
    ops.attention_merge(partials, merges, t, merged, heads, hd)
    got = ops.attention_merge_o(partials, merges, t, whole, weight, rows, heads, kv, hd)
    x = merged.double().view(t, kv, -1).transpose(0, 1).contiguous()
    w = weight.double().view(n, kv, -1).permute(1, 2, 0).contiguous()
    # (the merge's arithmetic is attention_merge's, so its bits; what is left is a float32 sum of heads / kv * head_dim products)
    bound = torch.bmm(x.abs(), w.abs()) * (heads // kv * hd) * 2.0 ** -24 + 1e-30
    assert ((got.double() - torch.bmm(x, w)).abs() <= bound).all() and got.isfinite().all()


def test_rule_and_refusals(ops):
    rows = ops.attention_merge_o_rows
    assert rows(1, 14, 2, 64, 896) == 1 and rows(2, 14, 2, 64, 896) == 2 and rows(ops.compute_units(), 14, 2, 64, 896) == 0
    assert rows(1, 34, 2, 64, 896) == 0 and rows(1, 14, 2, 96, 896) == 0 and rows(0, 14, 2, 64, 896) == 0 and rows(1, 16, 16, 128, 8192) == 0

    def call(heads=2, hd=64, cols=128, rows=1, n=8, dtype=torch.bfloat16):
        return ops.attention_merge_o(torch.zeros(heads * (hd + 2)).cuda(), torch.zeros(1, 4, dtype=torch.int32).cuda(), 1, torch.zeros(1, heads * hd, dtype=torch.bfloat16).cuda(),
                                     torch.ones(n, cols, dtype=dtype).cuda(), rows, heads, 1, hd)

    assert call().eq(0).all()
    for bad in (dict(rows=0), dict(rows=5), dict(hd=96, cols=192), dict(heads=17, cols=17 * 64), dict(cols=64), dict(dtype=torch.float32)):
        with pytest.raises(ops.KernelError):
            call(**bad)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, kv, hd, n, splits", [(14, 2, 64, 40, [65, 4]), (20, 2, 128, 24, [94, 5, 5]), (12, 1, 64, 9, [128]), (9, 1, 128, 8, [64, 0, 33])])
def test_more_records_than_a_wave_has_lanes(ops, dtype, heads, kv, hd, n, splits):
    """Sixty-four records are read at a time; the second head of a wave (groups of more than eight) asks for its own.  Against 64 bits: beyond 32 records the merge
    by itself adds up in another order."""
    t, g, slots = len(splits), torch.Generator().manual_seed(heads), sum(splits)
    records = torch.randn(slots, heads, hd + 2, generator=g)
    records[..., hd + 1] = records[..., hd + 1].abs() + 0.5
    merges = torch.tensor([(r, sum(splits[:r]), splits[r], 1) for r in range(t)], dtype=torch.int32).cuda()
    weight = torch.randn(n, heads * hd, generator=g).to(dtype).cuda()
    whole = torch.randn(t, heads * hd, generator=g).to(dtype)
    got = ops.attention_merge_o(records.reshape(-1).cuda(), merges, t, whole.cuda(), weight, 1, heads, kv, hd).double().cpu()
    x, off = whole.double().view(t, heads, hd), torch.zeros(t, heads, hd, dtype=torch.float64)
    for r, count in enumerate(splits):
        if count:
            mine = records[sum(splits[:r]):sum(splits[:r]) + count].double()
            share = torch.exp(mine[..., hd] - mine[..., hd].amax(0))
            denom = (share * mine[..., hd + 1]).sum(0)[:, None]
            x[r] = (share[..., None] * mine[..., :hd]).sum(0) / denom
            # (float32 sums of `count` products, their factors a few roundings each; then the heads' own rounding)
            off[r] = (share[..., None] * mine[..., :hd].abs()).sum(0) / denom * (count + 32) * 2.0 ** -23 + x[r].abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0)
    by_kv = lambda a: a.reshape(t, kv, -1).transpose(0, 1)
    w = weight.double().cpu().view(n, kv, -1).permute(1, 2, 0)
    bound = (by_kv(x.abs() + off) @ w.abs()) * (heads // kv * hd) * 2.0 ** -24 + by_kv(off) @ w.abs() + 1e-30
    assert ((got - by_kv(x) @ w).abs() <= bound).all()
