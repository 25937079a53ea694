"""The float32 product of few rows from a fragment-ordered copy, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops

    ops.load()
    return ops


def _operands(m, n, k):
    gen = torch.Generator().manual_seed(m * 131 + n * 7 + k)
    return (torch.randn((m, k), generator=gen).cuda(), (torch.randn((n, k), generator=gen) * 0.05).cuda(), torch.randn((n,), generator=gen).cuda())


def _bound(x, w, slices):
    """A value's rounding errors: at most 128 products one after the other, K / 128 such runs, 16 waves, the slices."""
    return (128 + x.shape[1] // 128 + 16 + slices + 2) * 2.0 ** -24 * (x.abs().double() @ w.abs().double().T)


# tiles of 1 to 4, rows of W that end inside a block and inside four neighbours, K of a few steps, one that sixteen waves hold, long ones whose steps
# are no multiple of what is under way; waves 4, 8, 16 whole and in slices whose last is shorter
@pytest.mark.parametrize("m,n,k,waves,slices", [
    (1, 16, 64, 8, 1), (3, 331, 896, 8, 1), (16, 37, 1024, 8, 1), (17, 128, 880, 8, 1), (33, 100, 1040, 8, 1), (64, 66, 1600, 8, 1),
    (2, 1152, 2048, 16, 1), (32, 50, 1040, 16, 1), (5, 130, 4112, 16, 1), (31, 18, 2064, 16, 1),
    (1, 70, 640, 4, 1), (4, 257, 2048, 4, 1), (48, 33, 1552, 4, 1), (64, 64, 4112, 4, 1),
    (1, 896, 4864, 8, 8), (4, 130, 1008, 8, 4), (20, 896, 896, 8, 4), (64, 48, 4880, 8, 8), (16, 35, 8192, 8, 8), (8, 64, 16, 8, 1)])
def test_against_float64(ops, m, n, k, waves, slices):
    x, w, bias = _operands(m, n, k)
    copy = ops.fragment_order(w)
    assert copy.shape == (n, k) and copy.data.dtype == torch.float32
    got = ops.gemm_fp32_stream(x, copy, waves + 256 * slices, bias if slices == 1 else None)
    assert got.shape == ((m, n) if slices == 1 else (slices, m, n))
    want = x.double() @ w.double().T
    total = got.double() - bias.double() if slices == 1 else got.double().sum(0)
    room = _bound(x, w, slices) + (2.0 ** -23 * (want + bias.double()).abs() if slices == 1 else 0)
    assert ((total - want).abs() <= room).all()
    # a row's sums say nothing about the other rows of its tile
    if m > 1 and (m - 1) // 16 == (m - 2) // 16:
        fewer = ops.gemm_fp32_stream(x[:m - 1].contiguous(), copy, waves + 256 * slices, bias if slices == 1 else None)
        assert torch.equal(fewer, got[..., :m - 1, :])


@pytest.mark.parametrize("m,n,k,waves", [(1, 6, 64, 8), (4, 9728, 896, 8), (17, 70, 1040, 16), (3, 150, 4096, 4), (64, 34, 2048, 4)])
def test_gate_and_up(ops, m, n, k, waves):
    x, w, _ = _operands(m, n, k)
    copy = ops.fragment_order(w)
    plain = ops.gemm_fp32_stream(x, copy, waves + 256)
    for act in ("silu", "gelu_tanh"):
        assert torch.equal(ops.gemm_fp32_stream(x, copy, waves + 256, act=act), ops.swiglu(plain, act=act))


def test_infinities_stay_in_their_row_and_steps_past_the_end_add_nothing(ops):
    x, w, _ = _operands(4, 40, 1040)  # 65 steps in eight waves of nine: the last wave has two
    x[1, 1039], x[2, 3], x[3, 500] = float("inf"), float("-inf"), float("nan")
    w = w.abs() + 1e-3
    for plan in (8 + 256, 16 + 256, 4 + 256, 8 + 256 * 3):
        y = ops.gemm_fp32_stream(x, ops.fragment_order(w), plan)
        y = y.sum(0) if y.ndim == 3 else y
        assert torch.isfinite(y[0]).all() and (y[1] == float("inf")).all() and (y[2] == float("-inf")).all() and torch.isnan(y[3]).all()


def test_refusals(ops):
    x, w, bias = _operands(4, 32, 64)
    copy = ops.fragment_order(w)
    for bad in (2 + 256, 8, 8 + 256 * 17, 8 + 256 * 5):  # no such waves, no slice, too many, more slices than steps
        with pytest.raises(ops.KernelError):
            ops.gemm_fp32_stream(x, copy, bad)
    with pytest.raises(ops.KernelError):  # a bias belongs to a whole product
        ops.gemm_fp32_stream(x, copy, 8 + 256 * 2, bias)
    with pytest.raises(ops.KernelError):  # sixteen waves: up to 32 rows
        ops.gemm_fp32_stream(torch.zeros((33, 64), device="cuda"), copy, 16 + 256)
    with pytest.raises(ops.KernelError):
        ops.fragment_order(w[:, :40].contiguous())
    assert ops.gemm_fp32_stream(x[:0], copy, 8 + 256).shape == (0, 32)


@pytest.mark.parametrize("m", [1, 2, 3, 16, 17, 33, 64, 65])
def test_linear_takes_the_copy(ops, m):
    """A layer's products with and without a copy: the same within the two ways' rounding, and whole where the kernel is not the better one."""
    from types import SimpleNamespace

    from from_scratch_inference_engine_amd.parts.linear import Linear

    x, w, bias = _operands(m, 896, 896)
    with_copy, without = Linear(896, 896, bias=True), Linear(896, 896, bias=True)
    for lin in (with_copy, without):
        lin.weight, lin.bias = w, bias
        lin.prepare(lin is with_copy)
    assert with_copy.streamed32 is not None and with_copy.streamed is None and without.streamed32 is None
    room = 2 * _bound(x, w, 8) + 2.0 ** -22
    assert ((with_copy(x).double() - without(x).double()).abs() <= room).all()
    for lin in (with_copy, without):
        lin.bias = None
    ctx = SimpleNamespace(partial_sums_ok=True)
    a, b = (y.double().sum(0) if y.ndim == 3 else y.double() for y in (with_copy.for_residual(x, ctx), without.for_residual(x, ctx)))
    assert ((a - b).abs() <= room).all()
    assert with_copy.for_residual(x, SimpleNamespace(partial_sums_ok=False)).ndim == 2
    assert with_copy.drop_copy() == 896 * 896 * 4 and with_copy.streamed32 is None
    with_copy.prepare()
    with_copy.weight = w.clone()
    assert with_copy.streamed32 is None
