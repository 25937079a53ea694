"""Which kernel, copy and slices a product of few rows takes, where a choice was measured to matter."""

import pytest
import torch

from from_scratch_inference_engine_amd.parts.linear import Linear


@pytest.mark.parametrize("n, k, rows, copy", [(2048, 2048, 16, True), (2048, 2048, 64, True), (2048, 2048, 65, False), (2048, 2048, 128, False),
                                              (4096, 2048, 17, True), (4096, 2048, 128, True)])
def test_copies_of_small_weights_are_for_sixty_four_rows(n, k, rows, copy):
    lin = Linear(k, n)
    lin.weight = torch.empty((n, k), dtype=torch.bfloat16, device="meta")
    assert lin.copy_for(rows) is None and lin.wide_weight(rows) is lin.weight
    lin.streamed = object()
    assert (lin.copy_for(rows) is lin.streamed) == copy and (lin.wide_weight(rows) is lin.weight) == (not copy)


@pytest.mark.parametrize("copies_from, size, copy", [(0, 64, True), (None, 64, True), (1 << 20, 1 << 20, False), (1 << 20, 2 << 20, True),
                                                     (48 << 20, 16 << 20, True)])
def test_copies_where_their_least_size_is_set(copies_from, size, copy, monkeypatch):
    monkeypatch.setattr(Linear, "streamed_copy_from", copies_from)
    lin = Linear(size // 2, 1)
    lin.weight = torch.empty((1, size // 2), dtype=torch.bfloat16, device="meta")
    lin.streamed = object()
    assert lin.copy_for(64) is lin.streamed
    assert (lin.copy_for(65) is lin.streamed) == copy and (lin.copy_for(128) is lin.streamed) == copy


@pytest.mark.parametrize("m, n, k", [(17, 1024, 768), (64, 9728, 640), (40, 512, 896), (128, 14336, 512)])
def test_partial_sums_of_a_short_k_are_not_taken(m, n, k):
    lin = Linear(k, n)
    lin.weight = torch.empty((n, k), dtype=torch.bfloat16, device="meta")
    assert lin.partial_sums(torch.empty((m, k), dtype=torch.bfloat16, device="meta")) is None


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k, cut", [(40, 896, 896, True), (64, 4096, 256, True), (32, 4096, 896, True), (64, 9728, 896, False),
                                          (80, 6144, 896, False), (128, 1024, 896, False), (40, 2048, 1024, True)])
def test_slices_of_a_short_k(m, n, k, cut):
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    assert (ops.gemm_mfma_wide_best_splits(m, n, k) > 1) == cut


@pytest.mark.parametrize("n, k, splits, wide", [
    (896, 896, 7, True), (1024, 1024, 8, True), (1536, 1536, 6, True), (4096, 768, 6, True), (896, 3072, 8, True), (512, 4096, 8, True),
    (3584, 896, 7, False), (1536, 1024, 8, False), (512, 2048, 8, False), (1536, 2048, 8, False), (2048, 640, 5, False)])
def test_few_rows_without_a_copy(n, k, splits, wide):
    assert Linear(k, n).slices_beat_few_rows(splits) == wide


@pytest.mark.gpu
@pytest.mark.parametrize("n, k, splits", [
    (896, 896, 7), (1536, 1536, 6), (896, 2048, 8), (1536, 2048, 8), (896, 3072, 8), (1536, 4096, 8), (896, 4864, 8), (2048, 2048, 8),
    (1536, 8192, 13), (2048, 8192, 13), (1024, 13824, 14), (4096, 8192, 8), (3584, 3584, 7), (6144, 2048, 4), (3584, 18944, 8)])
def test_slices_of_sixteen_rows(n, k, splits):
    """Up to eight slices, 14 of a long K: more cost the norm that adds them up more than the product gains."""
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    if ops.compute_units() == 256:
        assert ops.gemm_mfma_wide_best_splits(8, n, k) == splits


@pytest.mark.gpu
@pytest.mark.parametrize("k, short, long", [(512, 4, 0), (896, 7, 0), (1024, 8, 2), (1536, 6, 3), (2048, 8, 4), (3072, 8, 6)])
@pytest.mark.parametrize("rows", [1, 16])
def test_long_slices_for_those_who_pay_for_each(k, short, long, rows):
    """The sums of both cuts are the product's: within a float32 rounding of 2^-24 for each of K additions of each term."""
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)
    lin = Linear(k, 512)
    lin.weight = torch.randn((512, k), generator=torch.Generator().manual_seed(k)).to(torch.bfloat16).cuda()
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).cuda()
    exact, size = x.double() @ lin.weight.double().t(), x.double().abs() @ lin.weight.double().abs().t()
    for sums, slices in ((lin.partial_sums(x, few_rows=True), short), (lin.partial_sums(x, few_rows=True, long_slices=True), long)):
        if slices == 0:
            assert sums is None
            continue
        if ops.compute_units() == 256:
            assert sums.shape[0] == slices
        assert ((sums.double().sum(0) - exact).abs() <= k * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("n, k, whole", [(896, 896, False), (3584, 18944, False), (5120, 5120, False), (6144, 896, False), (4096, 14336, False),
                                         (4096, 2048, True), (8192, 8192, True), (3072, 1536, True), (3072, 2048, False)])
def test_float32_slices_of_few_rows(n, k, whole, monkeypatch):
    from from_scratch_inference_engine_amd.ops import functions

    monkeypatch.setattr(functions, "compute_units", lambda: 256)
    assert (functions.gemm_mfma_fp32_splits(k, n) == 1) == whole


@pytest.mark.parametrize("slices, timed, own", [(1, False, True), (1, True, False), (2, False, True), (2, True, True)])
def test_a_whole_product_of_many_rows_is_left_to_the_librarys_timed_kernels(slices, timed, own, monkeypatch):
    from from_scratch_inference_engine_amd import ops
    from from_scratch_inference_engine_amd.parts import linear

    class Ctx:
        partial_sums_ok = True

    monkeypatch.setattr(ops, "gemm_tile_plan", lambda *a: (2, slices))
    monkeypatch.setattr(ops, "gemm_mfma_tile", lambda *a, **kw: "sums")
    monkeypatch.setattr(linear, "library_tuning_enabled", lambda: timed)
    lin = Linear(18944, 64)
    lin.weight = torch.empty((64, 18944), dtype=torch.bfloat16, device="meta")
    assert (lin.residual_sums(torch.empty((256, 18944), dtype=torch.bfloat16, device="meta"), Ctx) == "sums") == own


@pytest.mark.gpu
@pytest.mark.parametrize("n, k", [(896, 4864), (896, 896), (2048, 2048), (5120, 5120), (512, 2048)])
def test_a_float32_row_of_a_prompt_does_not_depend_on_the_rows_beside_it(n, k):
    """Whole and as a residual projection in slices: the first rows of 700 are the bits that 70 and 300 of them give."""
    from from_scratch_inference_engine_amd import ops

    ops.load(build_if_missing=False)

    class Ctx:
        partial_sums_ok = True

    lin = Linear(k, n)
    lin.weight = torch.randn((n, k), generator=torch.Generator().manual_seed(n)).cuda()
    x = torch.randn((700, k), generator=torch.Generator().manual_seed(k)).cuda()
    whole, sums = lin(x), lin.for_residual(x, Ctx)
    for m in (70, 300):
        assert torch.equal(lin(x[:m].contiguous()), whole[:m])
        assert torch.equal(lin.for_residual(x[:m].contiguous(), Ctx), sums[..., :m, :])


@pytest.mark.parametrize("head, hidden, long", [(64, 896, False), (128, 640, False), (128, 512, True), (64, 256, True), (160, 896, True), (256, 2048, True)])
def test_slices_that_attention_adds_up(head, hidden, long):
    from types import SimpleNamespace

    from from_scratch_inference_engine_amd.parts.attention import GQAttention

    assert GQAttention.wants_long_slices.fget(SimpleNamespace(head_dim=head, qkv=Linear(hidden, 4 * head))) == long


def _block_plan(m, n, k, sums):
    from from_scratch_inference_engine_amd import ops

    return ops.load().fsie_gemm_mfma_block_plan(m, n, k, int(sums), 256)


@pytest.mark.parametrize("m, n, k, sums", [
    (129, 8192, 8192, False), (384, 8192, 8192, False), (384, 5120, 13824, False), (96, 27648, 5120, False), (128, 16384, 5120, False), (300, 14336, 8192, False),
    (100, 14336, 8192, True), (600, 5120, 13824, True),                                              # weights beyond what the estimate was fitted to
    (1845, 512, 6656, False), (2284, 432, 11776, False),                                             # x that every die reads
    (65, 10240, 2048, True),                                                                          # slices of more rows than the norm adds up quickly
    (200, 896, 900, False), (200, 900, 896, False), (0, 896, 896, False), (16 << 20, 896, 64, False), (200, 16 << 20, 64, False)])
def test_small_tiles_leave_to_the_library(m, n, k, sums):
    assert _block_plan(m, n, k, sums) == -1


@pytest.mark.parametrize("m, n, k, sums, plan", [
    (17, 768, 768, False, (0, 1)), (64, 512, 896, False, (3, 1)), (160, 8192, 2048, False, (1, 1)), (136, 6144, 4096, False, (1, 1)), (129, 8192, 2048, False, (1, 1)), (1375, 1152, 896, False, (1, 1)),
    (256, 16384, 2048, False, (2, 1)), (200, 16384, 5120, False, (2, 1)), (200, 16384, 8192, False, (2, 1)), (224, 8192, 8192, True, (2, 2)), (96, 896, 4864, True, (3, 7)), (192, 4096, 14336, True, (2, 4)), (1000, 3584, 3584, False, (2, 1))])
def test_small_tiles_take(m, n, k, sums, plan):
    got = _block_plan(m, n, k, sums)
    assert (got % 256, got // 256) == plan


@pytest.mark.parametrize("m, n, k, sums, plan", [
    (1375, 896, 4864, True, (2, 3)), (513, 2048, 8192, True, (2, 3)), (1700, 896, 4864, True, None),   # (the last: a whole product is as fast by the fit)
    (640, 3584, 3584, False, (2, 1)), (1025, 2048, 2048, False, (2, 1)),
    (319, 3584, 3584, False, None), (320, 3584, 3584, False, (1, 1)), (2601, 896, 4864, True, None), (400, 3584, 3584, True, None),
    (1375, 768, 4864, True, None), (700, 1024, 6144, False, (3, 1)), (1895, 1088, 11008, False, None)])
def test_small_tiles_of_middle_sizes(m, n, k, sums, plan):
    got = _block_plan(m, n, k, sums)
    assert (None if got < 0 else (got % 256, got // 256)) == plan


def test_plans_of_small_tiles_are_ones_the_kernel_takes():
    import random

    rng = random.Random(7)
    taken = 0
    for _ in range(4000):
        m, n, k = int(2 ** rng.uniform(0, 13)), 16 * int(2 ** rng.uniform(0, 13)), 64 * int(2 ** rng.uniform(0, 10))
        sums = rng.random() < 0.5
        got = _block_plan(m, n, k, sums)
        if got != -1:
            taken += 1
            tile, slices = got % 256, got // 256
            assert 0 <= tile <= 3 and 1 <= slices <= (8 if sums else 1) and slices <= k // 64, (m, n, k, sums)
    assert taken > 1000


def test_a_norm_whose_weight_does_not_lie_on_16_bytes_does_not_wait_for_its_product():
    from from_scratch_inference_engine_amd.parts.base import HiddenState
    from from_scratch_inference_engine_amd.parts.norm import RMSNorm

    norm, hidden = RMSNorm(64, 1e-6), HiddenState(torch.zeros(1, 64))
    room = torch.ones(64 + 8)
    aligned = (-room.data_ptr() // 4) % 4  # (values to the next 16 bytes)
    for off in range(4):
        norm.weight = room[aligned + off:aligned + off + 64]
        assert norm.can_wait(hidden, torch.bfloat16) == (off == 0)
    norm.weight = room[aligned:aligned + 64]
    for sums, waits in ((torch.zeros(3, 1, 64), True), (torch.zeros(1, 64, dtype=torch.bfloat16), False), (torch.zeros(3, 1, 64, dtype=torch.bfloat16), False)):
        hidden.delta = sums
        assert norm.can_wait(hidden, torch.bfloat16) == waits
    hidden.delta = None
    assert not norm.can_wait(hidden, torch.float32)
    hidden.delta_scale = 0.5
    assert not norm.can_wait(hidden, torch.bfloat16)


@pytest.mark.parametrize("rows, asked", [(1, 3), (2, 3), (3, 0), (40, 0)])
def test_only_steps_of_few_rows_ask_whether_a_norm_may_wait(rows, asked):
    """An eager step of many layers is bound by the host: a layer of more rows goes through its parts and nothing else (its rows are its shape's:
    the length of a tensor is four calls)."""
    from types import SimpleNamespace

    from from_scratch_inference_engine_amd.parts.base import HiddenState
    from from_scratch_inference_engine_amd.parts.block import PreNormBlock

    questions, order = [], []

    class Norm:
        def __call__(self, hidden, dtype):
            order.append("norm")
            return "x"

        def can_wait(self, hidden, dtype):
            questions.append(hidden)
            return False

    part = SimpleNamespace(forward=lambda x, ctx, *cache: order.append("part") or len(order))
    hidden = HiddenState(SimpleNamespace(shape=(rows, 8)))
    PreNormBlock(Norm(), part, Norm(), part).forward(hidden, SimpleNamespace(compute_dtype=torch.bfloat16, sums_in_one=False), None)
    assert order == ["norm", "part", "norm", "part"] and hidden.delta == 4 and len(questions) == asked


def test_the_merge_makes_the_output_projection_where_a_wave_has_one_head_or_tokens_are_few():
    """Every workgroup merges its kv head's records again: groups of more heads than a workgroup has waves are slower from three tokens on (float32:
    two), and beyond 12 heads."""
    from from_scratch_inference_engine_amd import ops
    from from_scratch_inference_engine_amd.ops.functions import dtype_code

    rows = lambda t, heads, kv, hd, n, dtype=torch.bfloat16: ops.load().fsie_attention_merge_o_rows(t, heads, kv, hd, n, dtype_code(dtype), 256)
    assert [rows(t, 14, 2, 64, 896) for t in (1, 2, 3, 4, 5)] == [1, 2, 3, 4, 0]
    assert [rows(t, 8, 1, 128, 1024) for t in (1, 4, 8)] == [1, 2, 4] and [rows(t, 8, 1, 128, 1024, torch.float32) for t in (1, 4, 8)] == [1, 2, 4]
    assert [rows(t, 12, 1, 128, 1536) for t in (1, 2, 3, 4)] == [1, 2, 0, 0] and [rows(t, 12, 1, 128, 1536, torch.float32) for t in (1, 2)] == [1, 0]
    assert rows(1, 16, 1, 128, 2048) == rows(2, 16, 1, 128, 2304) == rows(1, 13, 1, 64, 512) == 0
    assert rows(1, 14, 2, 96, 896) == rows(0, 14, 2, 64, 896) == 0
