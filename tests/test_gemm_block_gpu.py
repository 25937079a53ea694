"""The products of a hundred to some thousand rows in small tiles: against float64, at the edges of tiles, steps and slices."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from from_scratch_inference_engine_amd import ops as module

    module.load(build_if_missing=False)
    return module


# one step of K, fewer steps than stages, a last tile of one row and one of 16 of N, a whole number of tiles, more tiles than units
@pytest.mark.parametrize("m, n, k", [(65, 16, 64), (1, 48, 128), (129, 144, 192), (128, 256, 320), (300, 1152, 896), (513, 272, 1088), (1375, 896, 256)])
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_products_in_small_tiles(ops, m, n, k, tile):
    gen = torch.Generator().manual_seed(m + n + k)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).cuda() for s in ((m, k), (n, k)))
    bias = torch.randn(n, generator=gen).cuda()
    exact, bound = x.double() @ w.double().t(), k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    for add in (None, bias):
        want = exact if add is None else exact + add.double()
        got = ops.gemm_mfma_block(x, w, ops.GEMM_BLOCK_PLAIN, tile, bias=add).double()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2 * bound).all()  # one rounding to bfloat16
    for splits in sorted({1, 2, min(5, k // 64)}):
        if splits > k // 64:
            continue
        got = ops.gemm_mfma_block(x, w, ops.GEMM_BLOCK_SUMS, tile, splits)
        assert got.shape == (splits, m, n) and got.dtype == torch.float32
        assert ((got.double().sum(0) - exact).abs() <= bound).all(), splits
        cut = k // 64 * (splits - 1) // splits * 64  # the last slice holds its own part of K only
        last = x[:, cut:].double() @ w[:, cut:].double().t()
        assert ((got[-1].double() - last).abs() <= bound).all(), splits


@pytest.mark.parametrize("m, n, k", [(200, 896, 896), (300, 128, 512), (96, 896, 2048), (700, 512, 512), (30, 896, 512), (17, 512, 896), (64, 2048, 320)])
def test_linear_takes_them(ops, m, n, k, monkeypatch):
    """What ``Linear`` makes of them, with the bias in the product and as partial sums, is the library's within their roundings; rows that the
    kernel's loads cannot read go to the library."""
    from types import SimpleNamespace

    from from_scratch_inference_engine_amd.parts import linear

    seen, block = [], ops.gemm_mfma_block
    monkeypatch.setattr(ops, "gemm_mfma_block", lambda *a, **kw: (seen.append(a[2]), block(*a, **kw))[1])
    gen = torch.Generator().manual_seed(n)
    layer = linear.Linear(k, n, bias=True)
    layer.weight = torch.randn(n, k, generator=gen).to(torch.bfloat16).cuda()
    layer.bias = torch.randn(n, generator=gen).cuda()
    x = torch.randn(m, k, generator=gen).to(torch.bfloat16).cuda()
    exact = x.double() @ layer.weight.double().t()
    size = exact.abs() + layer.bias.double().abs() + k * 2.0 ** -24 * (x.double().abs() @ layer.weight.double().abs().t())
    assert ((layer(x).double() - exact - layer.bias.double()).abs() <= 2.0 ** -7 * size).all()
    plain = ops.gemm_block_plan(m, n, k, ops.GEMM_BLOCK_PLAIN) is not None
    assert (ops.GEMM_BLOCK_PLAIN in seen) == plain
    layer.bias, layer.has_bias = None, False
    delta = layer.for_residual(x, SimpleNamespace(partial_sums_ok=True))
    assert ((delta.double().sum(0) if delta.ndim == 3 else delta.double()) - exact).abs().le(2.0 ** -7 * size).all()
    large = m > 128 and ops.gemm_tile_plan(m, n, k, ops.GEMM_TILE_SUMS) is not None
    slices = 1 if large or m <= 64 else (ops.gemm_block_plan(m, n, k, ops.GEMM_BLOCK_SUMS) or (0, 1))[1]
    assert (ops.GEMM_BLOCK_SUMS in seen) == (slices > 1) and (not slices > 1 or delta.shape == (slices, m, n))
    seen.clear()
    wide = torch.zeros((m, k + 4), dtype=torch.bfloat16, device="cuda")
    odd = wide[:, 4:]
    odd.copy_(x)
    assert ((layer(odd).double() - exact).abs() <= 2.0 ** -7 * size).all() and not seen
    layer.bias = torch.zeros(n + 1, device="cuda")[1:].copy_(torch.randn(n, generator=gen))  # (four bytes off the 16 that the kernel loads)
    layer.has_bias = True
    assert ((layer(x).double() - exact - layer.bias.double()).abs() <= 2.0 ** -7 * (size + layer.bias.double().abs())).all() and not seen
