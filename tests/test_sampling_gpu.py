"""The choice of a token where the kernel's bins, lists and runs have their edges."""

import pytest
import torch

import plain_qwen2 as plain

pytestmark = pytest.mark.gpu

PARAMS = [(1.0, 0, 1.0), (0.7, 1, 1.0), (0.8, 3, 1.0), (1.3, 50, 1.0), (1.0, 0, 0.0), (1.0, 0, 1e-6), (0.7, 0, 0.5),
          (1.0, 0, 0.999999), (2.0, 40, 0.9), (0.5, 10 ** 9, 0.3), (1.0, 1, 0.5)]


def rows_of(kind, n, vocab):
    g = torch.Generator().manual_seed(vocab + len(kind))
    x = torch.randn((n, vocab), generator=g)
    if kind == "narrow":      # all within a thousandth
        return x * 1e-3 + 7.0
    if kind == "wide":        # most of them far below the bins' range
        return x * 60.0
    if kind == "equal":       # one bin cannot be told from another
        return torch.full_like(x, -3.25)
    if kind == "ties":        # a handful of values: more tokens in a bin than the list holds where the vocabulary is large
        return (x * 2).round() + 0.0  # (no negative zeros: the order of the keys tells them from zero)
    if kind == "coarse":      # hundreds of tokens of one value: more than are compared with each other
        return (x * 10).round() / 4 + 0.0
    if kind == "masked":      # a few tokens allowed, the others at -inf
        keep = torch.rand((n, vocab), generator=g) < 0.02
        keep[:, vocab // 2] = True
        return torch.where(keep, x, torch.tensor(float("-inf")))
    return x * 2.5


@pytest.mark.parametrize("kind", ["plain", "narrow", "wide", "equal", "ties", "coarse", "masked"])
@pytest.mark.parametrize("vocab", [1, 2, 63, 65, 2047, 4096, 16385, 40007])
def test_kept_sets_and_draws(kind, vocab):
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    cases = [(t, k, p, u) for t, k, p in PARAMS for u in (0.003, 0.4999, 0.99999)]
    logits = rows_of(kind, len(cases), vocab)
    dev = lambda v, dt: torch.tensor(v, dtype=dt).cuda()
    t, k, p, u = zip(*cases)
    args = (dev(t, torch.float32), dev(k, torch.int32), dev(p, torch.float32), dev(u, torch.float64))
    got = ops.sample(logits.cuda(), *args).cpu().tolist()
    assert got == ops.sample(logits.cuda(), *args).cpu().tolist()  # (nothing depends on the order of the threads)
    for i, (temp, top_k, top_p, number) in enumerate(cases):
        want = plain.sample(logits[i], temp, top_k, top_p, number)
        if got[i] != want:
            # the oracle's weights are float64, the kernel's float32 exponentials of at most 2^-22 relative error
            # (|logit difference| / temperature times 2^-24 and the function's own): a draw or an edge of the kept
            # set within that of a boundary may fall on its other side
            alt = {plain.sample(logits[i], temp, top_k, min(max(top_p + dp, 0.0), 1.0) if top_p < 1.0 else 1.0,
                                min(max(number + d, 0.0), 1.0 - 1e-12))
                   for d in (-1e-5, 0.0, 1e-5) for dp in (-1e-6, 0.0, 1e-6)}
            assert got[i] in alt, (kind, vocab, cases[i], got[i], want)


@pytest.mark.parametrize("vocab", [5000, 16500, 40007])  # (a workgroup a row, and rows shared by 64 of them)
@pytest.mark.parametrize("top_k, top_p", [(20, 0.9), (0, 0.9), (20, 1.0), (0, 1.0)])
def test_rows_that_are_no_numbers_end(vocab, top_k, top_p):
    """A NaN (at the first token, inside the row, and first and last of what a workgroup of a shared row has: 512 and 768
    tokens at these sizes), an infinite maximum and a row of -inf give some token of the vocabulary."""
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    rows = 8
    x = torch.randn((rows, vocab), generator=torch.Generator().manual_seed(0))
    x[0, 17] = float("nan")
    x[1, 99] = float("inf")
    x[2, :] = float("-inf")
    x[4, 0] = float("nan")
    x[5, 3072] = x[5, 1536] = float("nan")
    x[6, 767] = x[6, 511] = x[6, 768] = float("nan")
    x[7, :] = float("nan")
    ones = torch.ones(rows).cuda()
    out = ops.sample(x.cuda(), ones, torch.full((rows,), top_k, dtype=torch.int32).cuda(), top_p * ones,
                     torch.full((rows,), 0.5, dtype=torch.float64).cuda()).cpu()
    assert ((out >= 0) & (out < vocab)).all() and out[1] == 99


@pytest.mark.parametrize("vocab", [300, 5000, 16500])
@pytest.mark.parametrize("temperature", [float("inf"), 1e-45])
def test_weights_that_are_no_numbers_leave_the_maximum(vocab, temperature):
    """At a temperature whose inverse is zero a token at -inf weighs (-inf) * 0, at one whose inverse is infinite the
    largest weighs 0 * inf: no sum of the row is a number then, and the choice is the largest token."""
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    rows = 6
    g = torch.Generator().manual_seed(vocab)
    x = torch.randn((rows, vocab), generator=g)
    x = torch.where(torch.rand((rows, vocab), generator=g) < 0.5, x, torch.tensor(float("-inf")))
    for top_p in (0.1, 0.9, 1.0):
        out = ops.sample(x.cuda(), torch.full((rows,), temperature).cuda(), torch.zeros(rows, dtype=torch.int32).cuda(),
                         torch.full((rows,), top_p).cuda(), torch.linspace(0.0, 0.99, rows, dtype=torch.float64).cuda())
        assert out.cpu().tolist() == x.argmax(1).tolist()


@pytest.mark.parametrize("rows, vocab", [(1, 16500), (3, 16500), (20, 16500), (21, 16500), (41, 16500), (42, 16500), (50, 40007), (64, 40007), (1100, 16500)])
def test_a_row_does_not_depend_on_how_many_workgroups_share_it(rows, vocab):
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    g = torch.Generator().manual_seed(rows)
    x = (torch.randn((rows, vocab), generator=g) * 2.5).cuda()
    kinds = [(0.0, 0, 1.0), (1.0, 0, 1.0), (0.8, 50, 1.0), (0.7, 0, 0.9), (1.0, 200, 0.95)]
    t, k, p = zip(*[kinds[i % 5] for i in range(rows)])
    args = [torch.tensor(t).cuda(), torch.tensor(k, dtype=torch.int32).cuda(), torch.tensor(p).cuda(),
            torch.rand((rows,), generator=g, dtype=torch.float64).cuda()]
    got = ops.sample(x, *args)
    for i in sorted({0, rows // 2, rows - 1, min(rows - 1, 4)}):
        assert got[i] == ops.sample(x[i:i + 1].contiguous(), *[a[i:i + 1].contiguous() for a in args])[0]
    assert torch.equal(ops.sample(x), x.argmax(1).to(torch.int32))


@pytest.mark.parametrize("rows, vocab", [(3, 700), (20, 5000), (3, 16500), (50, 16500)])
@pytest.mark.parametrize("top_k, top_p", [(0, 1.0), (40, 1.0), (0, 0.8), (40, 0.8), (10 ** 6, 1.0)])
def test_thresholds_that_no_row_has_are_not_passed(rows, vocab, top_k, top_p, monkeypatch):
    """The sampler leaves out an array that says nothing, and the tokens are those that the arrays give."""
    from from_scratch_inference_engine_amd import SamplingParams, ops
    from from_scratch_inference_engine_amd.sampling.sampler import Sampler, uniforms_for

    ops.load(build_if_missing=False)
    x = (torch.randn((rows, vocab), generator=torch.Generator().manual_seed(rows)) * 2.5).cuda()
    params = [SamplingParams(0.0 if i == 1 else 0.9, top_k, top_p) for i in range(rows)]
    passed, sample = [], ops.sample
    monkeypatch.setattr(ops, "sample", lambda *a: (passed.append(a), sample(*a))[1])
    got = Sampler(5).sample(x, params, list(range(rows)), [3] * rows)
    assert (passed[0][2] is not None) == (0 < top_k < vocab) and (passed[0][3] is not None) == (top_p < 1.0)
    dev = lambda v, dt: torch.tensor(v, dtype=dt).cuda()
    assert got == sample(x, dev([p.temperature for p in params], torch.float32), dev([top_k] * rows, torch.int32),
                         dev([top_p] * rows, torch.float32), dev(list(uniforms_for(5, range(rows), [3] * rows)), torch.float64)).tolist()


@pytest.mark.parametrize("kind", ["plain", "narrow", "wide", "ties", "coarse", "masked"])
@pytest.mark.parametrize("rows, vocab", [(24, 16384), (24, 16385), (24, 40007), (150, 16447), (600, 16384)])
def test_shared_rows_choose_what_rows_alone_do(kind, rows, vocab):
    """Both forms weigh a token by the same float32 and differ by the rounding of float64 sums.  Shared rows have bins of
    their own (listed whole up to a top k of 1,024; cut into finer ones beyond 64 tokens, whose members are bisected beyond
    512; lists of more than 4,096 tokens go back to the other form; waves that keep more than a few tokens of a line settle them
    on the way), in 32 parts, in four and in one."""
    from from_scratch_inference_engine_amd import ops
    from from_scratch_inference_engine_amd.ops.functions import _stream, check

    lib = ops.load(build_if_missing=False)
    cases = [(t, k, p) for t, k, p in [(1.0, 1024, 1.0), (1.0, 1025, 1.0), (1.0, 1025, 0.9), (0.8, 1024, 0.9), (2.0, 6000, 0.95), (1.0, 9000, 1.0),
                                       (5.0, 0, 0.99), (30.0, 0, 0.5), (0.01, 0, 0.9), (0.0005, 40, 0.9), (0.7, 64, 1.0), (1.0, 0, 0.3)]]
    x = rows_of(kind, rows, vocab).cuda()
    t, k, p = zip(*[cases[i % len(cases)] for i in range(rows)])
    dev = lambda v, dt: torch.tensor(v, dtype=dt).cuda()
    t, k, p, u = dev(t, torch.float32), dev(k, torch.int32), dev(p, torch.float32), torch.linspace(0.001, 0.999, rows, dtype=torch.float64).cuda()
    size = lib.fsie_sample_workspace(rows, vocab, 1)
    work = torch.full((size,), 255, dtype=torch.uint8).cuda()
    alone, shared = torch.full((rows,), -1, dtype=torch.int32).cuda(), torch.full((rows,), -1, dtype=torch.int32).cuda()
    args = (x.data_ptr(), rows, vocab, t.data_ptr(), k.data_ptr(), p.data_ptr(), u.data_ptr())
    check(lib.fsie_sample(*args, alone.data_ptr(), _stream()))
    check(lib.fsie_sample_split(*args, 0, work.data_ptr(), shared.data_ptr(), _stream()))
    if ops.sample_takes_arrays(rows, vocab, True):  # (the parameters come with the launch instead)
        assert torch.equal(ops.sample(x, *[v.cpu().numpy() for v in (t, k, p, u)]), shared)
    assert size > 0 and ((alone >= 0) & (alone < vocab)).all()
    assert torch.equal(alone, shared)


# temperature, top k, top p, and the width of a bulk of tokens far below the maximum (0: none)
COLD = [(0.003, 0, 0.9, 0), (0.001, 50, 1.0, 0), (0.001, 50, 0.9, 0), (0.0003, 50, 0.9, 0), (0.0005, 3000, 0.9, 0), (1e-5, 0, 0.5, 0), (1e-5, 9000, 0.9, 0),
        (0.004, 2000, 0.3, 0), (0.0003, 2, 1.0, 0), (1e-20, 3, 0.9, 0)]
BULKS = [(1.0, 20000, 1.0, 0.35), (4.0, 0, 0.9, 0.35), (1.0, 20000, 0.9, 0.5), (4.0, 0, 0.6, 0.2), (1.0, 20000, 1.0, 0.2), (1.0, 20000, 0.9, 1.0)]


@pytest.mark.parametrize("cases, vocab", [(COLD, 152064), (COLD, 16385), (BULKS, 152064)], ids=["cold", "cold and few", "bulks"])
def test_lists_settle_cold_rows_and_thresholds_in_a_bulk(cases, vocab):
    """Rows whose weights fall to zero within a bin or two, and rows whose threshold lies where most tokens are, choose what they choose
    alone, and from their lists: not by the slow way that a row takes which its list does not settle (the tokens that a row's list got are the first
    number of its workspace; an empty or a full list settles nothing)."""
    from from_scratch_inference_engine_amd import ops
    from from_scratch_inference_engine_amd.ops.functions import _stream, check

    lib, rows = ops.load(build_if_missing=False), 2 * len(cases)
    g = torch.Generator().manual_seed(vocab)
    x = torch.randn((rows, vocab), generator=g) * 2.5
    for r in range(rows):
        if cases[r % len(cases)][3]:
            x[r] = torch.randn(vocab, generator=g) * cases[r % len(cases)][3]
            x[r, 77], x[r, 5] = 25.0, 20.0
    x = x.cuda()
    t, k, p, _ = zip(*[cases[i % len(cases)] for i in range(rows)])
    dev = lambda v, dt: torch.tensor(v, dtype=dt).cuda()
    t, k, p, u = dev(t, torch.float32), dev(k, torch.int32), dev(p, torch.float32), torch.linspace(0.001, 0.999, rows, dtype=torch.float64).cuda()
    size = lib.fsie_sample_workspace(rows, vocab, 1)
    work = torch.full((size,), 255, dtype=torch.uint8).cuda()
    alone, shared = torch.full((rows,), -1, dtype=torch.int32).cuda(), torch.full((rows,), -1, dtype=torch.int32).cuda()
    args = (x.data_ptr(), rows, vocab, t.data_ptr(), k.data_ptr(), p.data_ptr(), u.data_ptr())
    check(lib.fsie_sample(*args, alone.data_ptr(), _stream()))
    check(lib.fsie_sample_split(*args, 0, work.data_ptr(), shared.data_ptr(), _stream()))
    assert torch.equal(alone, shared)
    listed = work.view(rows, -1)[:, :4].contiguous().view(torch.int32).flatten().tolist()
    assert all(0 < n <= 4096 for n in listed), listed


@pytest.mark.parametrize("rows, vocab, top_k, top_p, shared", [
    (16, 16384, 1, 0, 1), (40, 16384, 1, 0, 0), (256, 16384, 1, 0, 0), (300, 16384, 1, 0, 1), (40, 16384, 0, 1, 1), (100, 16384, 0, 1, 0), (300, 16384, 0, 1, 1),
    (40, 32000, 1, 0, 1), (100, 32000, 1, 0, 0), (160, 32000, 0, 1, 1), (224, 152064, 1, 0, 1), (256, 152064, 0, 1, 1), (96, 32000, 0, 0, 1), (100, 32000, 0, 0, 0),
    (128, 152064, 0, 0, 1), (160, 152064, 0, 0, 0), (300, 16384, 0, 0, 0), (4096, 16384, 1, 1, 1), (4097, 16384, 1, 1, 0), (8, 16383, 1, 1, 0), (0, 16384, 1, 1, 0)])
def test_rows_are_shared_where_that_is_faster(rows, vocab, top_k, top_p, shared):
    from from_scratch_inference_engine_amd import ops

    lib = ops.load(build_if_missing=False)
    assert lib.fsie_sample_shares(rows, vocab, top_k, top_p) == shared
    assert not shared or lib.fsie_sample_workspace(rows, vocab, top_k or top_p) > 0
