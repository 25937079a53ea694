"""What the ops say of arguments that are none: before anything is launched, and without a GPU."""

import pytest
import torch

from from_scratch_inference_engine_amd import ops


@pytest.mark.parametrize("x", [None, [[1.0]], torch.zeros(1, 128).numpy(), torch.zeros(1, 128, dtype=torch.bfloat16)])
def test_gate_and_up_of_something_else_than_a_gpu_tensor_is_refused(x):
    weight = torch.zeros(4, 128, dtype=torch.bfloat16)
    for norm in (None, (None, torch.zeros(128), 1e-6, None)):
        with pytest.raises(ops.KernelError, match="must be a tensor on the GPU"):
            ops.gemm_mfma_wide_swiglu(x, weight, norm=norm) if norm else ops.gemm_mfma_wide_swiglu(x, weight)
