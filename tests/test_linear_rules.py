"""Which kernel, copy and slices a product of few rows takes, where a choice was measured to matter."""

import pytest
import torch

from from_scratch_inference_engine_amd.parts.linear import Linear


@pytest.mark.parametrize("n, k, rows, copy", [(2048, 2048, 16, True), (2048, 2048, 17, False), (2048, 2048, 128, False),
                                              (4096, 2048, 17, True), (4096, 2048, 128, True)])
def test_copies_of_small_weights_are_for_sixteen_rows(n, k, rows, copy):
    lin = Linear(k, n)
    lin.weight = torch.empty((n, k), dtype=torch.bfloat16, device="meta")
    assert lin.copy_for(rows) is None and lin.wide_weight(rows) is lin.weight
    lin.streamed = object()
    assert (lin.copy_for(rows) is lin.streamed) == copy and (lin.wide_weight(rows) is lin.weight) == (not copy)
