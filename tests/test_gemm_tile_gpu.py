"""The product for many rows at the edges of its tiles, its stages and its slices."""

import pytest
import torch

import from_scratch_inference_engine_amd.ops as ops

# rows and columns of a workgroup of each tile
TILES = {0: (128, 256), 1: (256, 192), 2: (256, 256), 3: (256, 320)}


def operands(m, n, k):
    g = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    return ((torch.randn((m, k), generator=g)).to(torch.bfloat16).cuda(),
            (torch.randn((n, k), generator=g) * 0.1).to(torch.bfloat16).cuda())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("k", [64, 128, 192, 1088])
def test_partial_sums_at_the_edges(tile, k):
    """Rows and columns at, below and beyond a tile's; one step, an odd and an even number; uneven slices."""
    ops.load(build_if_missing=False)
    rows, cols = TILES[tile]
    for m, n in ((1, 16), (rows - 1, cols), (rows, cols + 16), (rows + 1, cols - 16), (2 * rows + 17, 2 * cols + 48)):
        x, w = operands(m, n, k)
        want = x.double() @ w.double().t()
        # products of 8-bit significands are exact in float32; a sum of k of them in any order is off by at most
        # k rounding errors of 2^-24 of the sum of their magnitudes
        bound = (k * 2.0 ** -24) * (x.double().abs() @ w.double().abs().t())
        for slices in sorted({1, min(2, k // 64), min(5, k // 64), min(16, k // 64)}):
            got = ops.gemm_mfma_tile(x, w, splits=slices, tile=tile)
            assert got.shape == (slices, m, n)
            assert ((got.double().sum(0) - want).abs() <= bound + 1e-30).all(), (tile, k, m, n, slices)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu", "clipped"])
def test_gate_and_up(tile, act):
    ops.load(build_if_missing=False)
    rows, cols = TILES[tile]
    kind = ops.GateAct("clipped", 2.0, 1.7) if act == "clipped" else ops.gate_act(act)
    for m, n, k in ((rows + 3, cols + 32, 320), (33, 16, 64), (2 * rows, 2 * cols, 128)):
        x, w = operands(m, n, k)
        d = (x.double() @ w.double().t()).to(torch.bfloat16).float()  # gate and up are rounded before they are multiplied
        want = ops.swiglu(d, act=kind).double()
        got = ops.gemm_mfma_tile_gated(x, w, act=kind, tile=tile).double()
        # the sums differ by rounding (as above), which may take gate or up to the next 8-bit value on either side (2^-7 of
        # it; an activation's slope is at most 1.7 (|u| + 1) here), and the result is rounded to 8 bits
        slack = 2.0 * (k * 2.0 ** -24) * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -7 * d.abs()
        slack = 1.7 * (slack[:, 0::2] * (d[:, 1::2].abs() + 1) + slack[:, 1::2] * (d[:, 0::2].abs() + 1))
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + slack + 1e-6).all(), (tile, act, m, n, k)
        # and such steps are rare: the bound on a sum is far below the distance of two 8-bit values
        assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.gpu
def test_replays_give_the_same_bits():
    ops.load(build_if_missing=False)
    x, w = operands(700, 1040, 640)
    first = ops.gemm_mfma_tile(x, w, splits=3, tile=2)
    for _ in range(5):
        assert torch.equal(first, ops.gemm_mfma_tile(x, w, splits=3, tile=2))


@pytest.mark.gpu
def test_sizes_it_does_not_take_are_refused():
    ops.load(build_if_missing=False)
    for m, n, k in ((10, 24, 64), (10, 32, 96)):
        x, w = operands(m, n, k)
        with pytest.raises(ops.KernelError):
            ops.gemm_mfma_tile(x, w)
    x, w = operands(10, 32, 128)
    with pytest.raises(ops.KernelError):
        ops.gemm_mfma_tile(x, w, splits=3)


def test_plan_names_a_tile_and_slices_that_the_kernel_takes():
    lib = ops.load(build_if_missing=False)
    plan = lib.fsie_gemm_mfma_tile_plan
    for m in (129, 200, 256, 511, 978, 2048, 4096, 16384):
        for n, k in ((37888, 3584), (9728, 896), (16384, 2048), (3584, 18944), (5120, 27648), (896, 4864), (2048, 8192), (48, 16384)):
            for result in (1, 2):
                got = plan(m, n, k, result, 256)
                if got >= 0:
                    assert got % 256 in TILES and 1 <= got // 256 <= k // 64 and (result == 2 or got // 256 == 1)
    assert plan(2048, 37888, 3584, 1, 256) >= 0 and plan(2048, 3584, 18944, 2, 256) >= 0  # a prompt at the 7B sizes
    assert plan(144, 16384, 2048, 1, 256) == -1      # too few tiles for the chip
    assert plan(2048, 2048, 8192, 2, 256) == -1      # the library cuts nothing there
    for n, k in ((37880, 3584), (37888, 3592)):      # rows that the stores or the steps of K do not fit
        assert plan(2048, n, k, 1, 256) == -1
    assert plan(2048, 1 << 20, 4096, 1, 256) == -1   # beyond the 32-bit offsets


def test_plan_deals_the_columns_of_tiles_to_eight_dies():
    """A die has an eighth of the units and gets every eighth column with all of its tiles: no plan whose fullest die takes
    more rounds than another plan's, at the same work a round."""
    plan = ops.load(build_if_missing=False).fsie_gemm_mfma_tile_plan
    assert plan(850, 1536, 18944, 2, 256) == 1 + 256 * 8    # (six slices of 128 x 256: 36 columns, 35 workgroups for 32 units)
    assert plan(1500, 3584, 18944, 2, 256) == 1 + 256 * 2   # (three of 256 x 256: 42 columns, 36 workgroups)
    assert plan(700, 3584, 18944, 2, 256) == 1 + 256 * 4
    assert plan(3000, 768 * 8, 768, 1, 256) == 1 + 256      # (20 columns of 256 x 320, 36 workgroups)
    for m, n, k in ((3000, 5120, 27648), (1500, 8192, 18944), (3000, 4096, 20480), (4096, 1024, 16384), (2048, 2048, 16384)):
        assert plan(m, n, k, 2, 256) == -1                  # the library fills the chip by itself
    assert plan(4096, 3584, 18944, 2, 256) >= 0 and plan(1024, 1024, 16384, 2, 256) >= 0


def test_plan_of_many_tiles_is_one_round():
    """Sums from half as many tiles as units on: one round of workgroups, or the library's product."""
    plan = ops.load(build_if_missing=False).fsie_gemm_mfma_tile_plan
    for m, n, k in ((2816, 3584, 18944), (3328, 3584, 18944), (2304, 4096, 18944), (2816, 4096, 18944), (2304, 5120, 27648), (1128, 8192, 28672)):
        assert plan(m, n, k, 2, 256) == -1
    assert plan(2560, 3584, 18944, 2, 256) == 3 + 256 * 2 and plan(2048, 5120, 27648, 2, 256) == 3 + 256 * 2
    assert plan(2048, 4096, 18944, 2, 256) == 2 + 256 * 2   # 128 tiles
