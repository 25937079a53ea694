"""The hand-written kernels as functions over torch tensors.

Each function checks on the host that the operands have the shapes, types and contiguity that the
kernel and its grid assume, then queues the kernel on torch's current stream.  Nothing here
computes with torch; a missing kernel library is an error, not a reason to fall back.
"""

from .functions import (FragmentOrdered, attention_merge, attention_mfma, attention_mfma_lds, attention_mfma_lds_ok,
                        attention_mfma_max_waves, attention_mfma_qkv, attention_mfma_qkv_ok, attention_mfma_qkv_o_rows, attention_merge_o, attention_merge_o_rows, attention_f32_qkv_ok, attention_mfma_rows, attention_scalar,
                        attention_tile_tokens, bias_add, compute_units, dtype_code, embedding, fragment_order, gemm, gemm_mfma_fp32, gemm_mfma_fp32_sums, gemm_mfma_fp32_splits, gemm_fp32_gated, gemm_fp32_tile, gemm_fp32_tile_splits, gemm_fp32_stream, gemm_fp32_stream_plan, GEMM_FP32_WHOLE, GEMM_FP32_GATED, GEMM_FP32_SUMS, gemm_mfma_skinny,
                        gemm_mfma_skinny_rope, gemm_mfma_wide, gemm_mfma_wide_best_splits, gemm_mfma_wide_splits_ok,
                        gemm_mfma_wide_swiglu, gemm_mfma_wide_takes, gemm_mfma_stream, gemm_mfma_block, gemm_block_plan, GEMM_BLOCK_PLAIN, GEMM_BLOCK_SUMS, gemm_mfma_normed, gemm_normed_takes, gemm_stream_plan, GEMM_STREAM_SUMS, GEMM_STREAM_GATED, GEMM_STREAM_POINT, GEMM_STREAM_PLAN_ACT, GEMM_STREAM_PLAN_ONE, random_fill,
                        residual_add,
                        rmsnorm, rmsnorm_plain, rope_kv_write, rope_table, sample, sample_takes_arrays, swiglu, zero_pages, zero_rows, zero_rows_of,
                        gate_act_code, gate_act, GateAct, gated_headnorm, gla_chunked, gla_scan, gla_step, gla_step_takes, head_gemm, latent_prep, rope_pairs, sandwich_norm, softcap,
                        stream_out, round_columns, gemm_mfma_skinny_gated, attention_prep, gate_heads, layer_norm, pair_embedding,
                        group_rmsnorm, causal_conv, mlstm_state_floats, mlstm_scan, mlstm_out, moe_route, moe_group, moe_gemm, moe_combine, moe_tile_rows, sum_round, bias_act, query_temperature, PointAct, NO_ACT, gemm_mfma_skinny_act, gemm_mfma_wide_act, gemm_mfma_wide_act_takes,
                        gemm_mfma_tile, gemm_mfma_tile_gated, gemm_tile_plan, GEMM_TILE_PAIR, GEMM_TILE_SUMS, pool_blocks, scaled_sum, round_to, GEMM_AUTO, GEMM_TILED, GEMM_SKINNY, GEMM_NARROW)
from .library import KernelError, KernelLibraryMissing, load
from .tuning import disable_library_tuning, enable_library_tuning, library_mm, library_tuning_enabled

__all__ = ["FragmentOrdered", "KernelError", "KernelLibraryMissing", "attention_merge", "attention_mfma", "attention_mfma_lds",
           "attention_mfma_lds_ok", "attention_mfma_max_waves", "attention_mfma_qkv", "attention_mfma_qkv_ok", "attention_mfma_qkv_o_rows", "attention_merge_o", "attention_merge_o_rows", "attention_f32_qkv_ok", "attention_mfma_rows", "attention_scalar",
           "attention_tile_tokens", "bias_add", "compute_units", "disable_library_tuning", "dtype_code", "embedding",
           "enable_library_tuning", "fragment_order", "gemm", "gemm_mfma_fp32", "gemm_mfma_fp32_sums", "gemm_mfma_fp32_splits", "gemm_fp32_gated", "gemm_fp32_tile", "gemm_fp32_tile_splits", "gemm_fp32_stream", "gemm_fp32_stream_plan", "GEMM_FP32_WHOLE", "GEMM_FP32_GATED", "GEMM_FP32_SUMS", "gemm_mfma_skinny", "gemm_mfma_skinny_rope", "gemm_mfma_wide",
           "gemm_mfma_tile", "gemm_mfma_tile_gated", "gemm_mfma_stream", "gemm_mfma_block", "gemm_block_plan", "GEMM_BLOCK_PLAIN", "GEMM_BLOCK_SUMS", "gemm_mfma_normed", "gemm_normed_takes", "gemm_stream_plan", "GEMM_STREAM_SUMS", "GEMM_STREAM_GATED", "GEMM_STREAM_POINT", "GEMM_STREAM_PLAN_ACT", "GEMM_STREAM_PLAN_ONE", "gemm_tile_plan", "gemm_mfma_wide_best_splits", "gemm_mfma_wide_splits_ok", "gemm_mfma_wide_swiglu", "gemm_mfma_wide_takes", "library_mm", "library_tuning_enabled", "load", "random_fill", "residual_add",
           "rmsnorm", "rmsnorm_plain", "rope_kv_write", "rope_table", "sample", "sample_takes_arrays", "swiglu", "zero_pages", "zero_rows", "zero_rows_of",
           "gate_act_code", "gate_act", "GateAct", "stream_out", "round_columns", "gemm_mfma_skinny_gated", "gla_chunked", "gated_headnorm", "gla_scan", "gla_step", "gla_step_takes", "head_gemm", "latent_prep", "rope_pairs", "sandwich_norm", "softcap",
           "attention_prep", "gate_heads", "layer_norm", "pair_embedding",
           "group_rmsnorm", "causal_conv", "mlstm_state_floats", "mlstm_scan", "mlstm_out", "moe_route", "moe_group", "moe_gemm", "moe_combine", "moe_tile_rows", "sum_round", "bias_act", "query_temperature", "PointAct", "NO_ACT",
           "gemm_mfma_skinny_act", "gemm_mfma_wide_act", "gemm_mfma_wide_act_takes", "pool_blocks", "scaled_sum", "round_to", "GEMM_AUTO", "GEMM_TILED", "GEMM_SKINNY", "GEMM_NARROW"]
