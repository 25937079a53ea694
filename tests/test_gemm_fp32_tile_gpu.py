"""The 32-bit product for many rows at the edges of its tiles, steps, runs and slices."""

import pytest
import torch

import from_scratch_inference_engine_amd.ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4, 28, 32, 36, 256, 260, 1100])
@pytest.mark.parametrize("m,n", [(65, 1), (64, 64), (63, 65), (129, 130), (200, 3)])
def test_against_64_bits(m, n, k):
    ops.load(build_if_missing=False)
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    bias = torch.randn((n,), generator=g).cuda()
    want = x.double() @ w.double().t()
    # a product and a sum of k of them in float32, in any order: at most k + 1 roundings of 2^-24 of the magnitudes' sum
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + bias.double().abs())
    assert ((ops.gemm_fp32_tile(x, w).double() - want).abs() <= bound).all()
    assert ((ops.gemm_fp32_tile(x, w, bias).double() - (want + bias.double())).abs() <= bound).all()
    for slices in range(2, 6):
        run = -(-k // slices)
        if -(-run // 32) * 32 * (slices - 1) >= k:
            with pytest.raises(ops.KernelError):
                ops.gemm_fp32_tile(x, w, splits=slices)
            continue
        got = ops.gemm_fp32_tile(x, w, splits=slices)
        assert got.shape == (slices, m, n) and ((got.double().sum(0) - want).abs() <= bound).all()


@pytest.mark.parametrize("k", [32, 64, 224, 256, 288, 1088])
@pytest.mark.parametrize("m,n", [(65, 48), (300, 130), (700, 1664)])  # few workgroups and more than 256 of them
def test_whole_steps_have_the_bits_of_the_others(m, n, k):
    """K of whole steps goes straight to LDS, four more columns of zeros take the kernel whose loads go through registers: the same sums in the same order."""
    ops.load(build_if_missing=False)
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    bias = torch.randn((n,), generator=g).cuda()
    more = [torch.nn.functional.pad(a, (0, 4)) for a in (x, w)]
    assert torch.equal(ops.gemm_fp32_tile(x, w), ops.gemm_fp32_tile(*more))
    assert torch.equal(ops.gemm_fp32_tile(x, w, bias), ops.gemm_fp32_tile(*more, bias))
    assert torch.equal(ops.gemm_fp32_gated(x, w, "silu"), ops.gemm_fp32_gated(*more, "silu"))
    if k == 1088:  # (slices of 512 and 768 values, with the four zeros as without)
        for slices in (3, 2):
            assert torch.equal(ops.gemm_fp32_tile(x, w, splits=slices), ops.gemm_fp32_tile(*more, splits=slices))


def test_slices_are_ones_the_kernel_takes():
    ops.load(build_if_missing=False)
    for m in (65, 200, 682, 2048):
        for n, k in ((896, 4864), (896, 896), (3584, 18944), (64, 256), (64, 300), (16, 512), (40, 2000)):
            slices = ops.gemm_fp32_tile_splits(m, n, k)
            assert 1 <= slices <= 16
            if slices > 1:
                x, w = torch.zeros((m, k), device="cuda"), torch.zeros((n, k), device="cuda")
                assert ops.gemm_fp32_tile(x, w, splits=slices).shape[0] == slices


@pytest.mark.parametrize("m", [3, 16, 17, 64])
@pytest.mark.parametrize("n,k", [(896, 896), (40, 448), (17, 4864), (64, 452), (896, 2000)])
def test_few_rows_in_slices(m, n, k):
    ops.load(build_if_missing=False)
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    want = x.double() @ w.double().t()
    bound = (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for slices in {2, 3, ops.gemm_mfma_fp32_splits(k)} - {1}:
        got = ops.gemm_mfma_fp32_sums(x, w, slices)
        assert got.shape == (slices, m, n) and ((got.double().sum(0) - want).abs() <= bound).all()


def test_slices_of_few_rows_are_never_empty():
    for k in list(range(4, 1200, 4)) + [4864, 8192, 18944]:
        slices, steps = ops.gemm_mfma_fp32_splits(k), -(-k // 16)
        assert 1 <= slices <= 8 and -(-steps // slices) * (slices - 1) < steps


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m, n, k", [(3, 34, 100), (4, 9728, 896), (16, 18, 2052), (17, 64, 300), (33, 130, 512), (64, 66, 1000), (65, 34, 260),
                                     (200, 130, 36)])
def test_gate_and_up_multiplied_in_the_epilogue(m, n, k, act):
    """The same bits as the product and the pass that multiplies, at the edges of the tiles of rows and of blocks of W."""
    ops.load(build_if_missing=False)
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    product = ops.gemm_mfma_fp32(x, w) if m <= 64 else ops.gemm_fp32_tile(x, w)
    assert torch.equal(ops.gemm_fp32_gated(x, w, act), ops.swiglu(product, act=act))
