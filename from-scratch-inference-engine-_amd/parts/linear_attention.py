"""Gated linear attention: a recurrent mixer whose cache is a state of fixed size per request."""

from __future__ import annotations

from typing import Dict, Optional

import torch

from .. import ops
from ..cache.manager import StateNeed
from .base import Mixer, ParamDecl, register_part
from .linear import Linear


@register_part("mixer", "gated_linear_attention")
class GatedLinearAttention(Mixer):
    """Per head a state S [key_dim, value_dim] in float32 that every token updates and reads:

        S_t = diag(alpha_t) S_(t-1) + k_t v_t^T,    o_t = S_t^T q_t,

    q = (W_q x) key_dim^(-1/2), k = W_k x, v = W_v x, and a decay per key channel
    alpha = sigmoid(W_a2 (W_a1 x) + b)^(1/tau) through a low rank.  Every head's o is RMS-normed over its
    value columns (one weight, shared by the heads), multiplied by act(W_g x) and projected by W_o.

    The projections that read x are one matrix (q, k, v, g rows one after the other; in steps of one token a request W_a1's rows
    too, and one kernel takes it from there to the output projection where it knows the sizes: ``ops.gla_step``).  The state lives in the
    cache manager's per-request slots: zero when a request starts, carried from step to step.  Steps with portions of prompts go
    chunk by chunk (``ops.gla_scan``, which then multiplies by W_a2 itself), others token by token.
    The decays, the state and the sums are float32 whatever the activations' type."""

    graph_safe = True  # the step's requests and slots are read from the device tables

    def __init__(self, hidden_size: int, n_heads: int, key_dim: int, value_dim: int, decay_rank: int, tau: float,
                 norm_eps: float, gate_activation: str = "silu"):
        if key_dim > 256:
            raise ValueError(f"gated linear attention: {key_dim} key channels a head are more than the kernel takes (256)")
        if not tau > 0:
            raise ValueError(f"gated linear attention: tau {tau} must be positive")
        ops.gate_act_code(gate_activation)
        self.hidden_size, self.n_heads, self.key_dim, self.value_dim = hidden_size, n_heads, key_dim, value_dim
        self.decay_rank, self.tau, self.norm_eps, self.gate_activation = decay_rank, float(tau), float(norm_eps), gate_activation
        self.k_width, self.v_width = n_heads * key_dim, n_heads * value_dim
        self.qkvg = Linear(hidden_size, 2 * self.k_width + 2 * self.v_width)
        self.a1 = Linear(hidden_size, decay_rank)
        self.a2 = Linear(decay_rank, self.k_width, bias=True)
        self.o = Linear(self.v_width, hidden_size)
        self.norm_weight = None
        self.in_proj: Optional[Linear] = None  # qkvg and a1 as one matrix, where steps of single tokens take both at once

    def param_decls(self) -> Dict[str, ParamDecl]:
        return {"qkvg_weight": ParamDecl((2 * self.k_width + 2 * self.v_width, self.hidden_size)),
                "a1_weight": ParamDecl((self.decay_rank, self.hidden_size)),
                "a2_weight": ParamDecl((self.k_width, self.decay_rank)),
                "a2_bias": ParamDecl((self.k_width,), "vector", "bias"),
                "norm_weight": ParamDecl((self.value_dim,), "vector", "norm"),
                "o_weight": ParamDecl((self.hidden_size, self.v_width))}

    def _set(self, part: Linear, weight) -> None:
        part.weight = weight
        self.in_proj = None  # (made of both matrices by ``prepare``)

    qkvg_weight = property(lambda s: s.qkvg.weight, lambda s, t: s._set(s.qkvg, t))
    a1_weight = property(lambda s: s.a1.weight, lambda s, t: s._set(s.a1, t))
    a2_weight = property(lambda s: s.a2.weight, lambda s, t: setattr(s.a2, "weight", t))
    a2_bias = property(lambda s: s.a2.bias, lambda s, t: setattr(s.a2, "bias", t))
    o_weight = property(lambda s: s.o.weight, lambda s, t: setattr(s.o, "weight", t))

    def prepare(self, device, compute_dtype) -> None:
        copies = bool(self.options.get("weight_copies", True))
        self.o.prepare(copies)
        self.in_proj = None
        n, k, rank = self.qkvg.out_features, self.hidden_size, self.decay_rank
        w = self.qkvg.weight
        if not (w is not None and self.a1.weight is not None and w.is_cuda and w.dtype == torch.bfloat16 and k % 8 == 0 and n % 16 == 0
                and ops.gla_step_takes(self.n_heads, self.key_dim, self.value_dim, rank)):
            self.qkvg.prepare(copies)
            return
        # a1's rows behind those of q, k, v and g: the two weights, and the copy of the first, become views of the whole
        both = Linear(k, n + rank)
        both.weight = torch.cat([w, self.a1.weight])
        self.qkvg.weight, self.a1.weight = both.weight[:n], both.weight[n:]
        both.prepare(copies)
        if both.streamed is not None:
            self.qkvg.streamed = ops.FragmentOrdered(both.streamed.data[:n * k], n, k)
        self.in_proj = both

    def release_optional_memory(self) -> int:
        freed = self.qkvg.drop_copy()
        return self.o.drop_copy() + (freed if self.in_proj is None else self.in_proj.drop_copy())

    def cache_need(self) -> StateNeed:
        return StateNeed((self.n_heads, self.key_dim, self.value_dim), "float32")

    def forward(self, x: torch.Tensor, ctx, cache) -> torch.Tensor:
        if self.in_proj is not None and x.dtype == torch.bfloat16 and 0 < x.shape[0] == ctx.seq_slots.shape[0]:
            # one token a request: one product, one kernel from there to the output projection (8 requests of 8 heads of 128 x 256
            # at hidden size 2,048, a layer, us: products 9.2, 5.5 and 3.6, operands 3.7, update 7.5, norm and gate 4.0 before)
            p, kw, vw = self.in_proj(x), self.k_width, self.v_width
            y = ops.gla_step(p, 0, kw, 2 * kw, 2 * kw + vw, 2 * kw + 2 * vw, self.a2.weight, self.a2.bias, cache.state, ctx.q_starts,
                             ctx.seq_slots, self.norm_weight, self.n_heads, self.key_dim, self.value_dim, self.key_dim ** -0.5,
                             1.0 / self.tau, self.norm_eps, self.gate_activation)
            return self.o.for_residual(y, ctx)
        p = self.qkvg(x)
        a, a2 = self.a1(x), self.a2.weight
        z, bottleneck = None, None
        if (a.dtype == torch.bfloat16 and self.decay_rank % 32 == 0 and ops.gla_chunked(x.shape[0], ctx.seq_slots.shape[0])
                and a.is_contiguous() and a2.is_contiguous() and a.data_ptr() % 16 == 0 and a2.data_ptr() % 16 == 0):
            bottleneck = (a, a2, self.a2.bias)  # (the scan's first kernel multiplies)
        else:
            z = self.a2(a, out_dtype=torch.float32)  # the decays before the sigmoid, bias added, float32 from here on
        o = ops.gla_scan(p, 0, self.k_width, 2 * self.k_width, z, cache.state, ctx.q_starts, ctx.seq_slots, self.n_heads,
                         self.key_dim, self.value_dim, self.key_dim ** -0.5, 1.0 / self.tau, bottleneck=bottleneck)
        y = ops.gated_headnorm(o, p[:, 2 * self.k_width + self.v_width:], self.norm_weight, self.norm_eps, self.n_heads,
                               self.gate_activation)
        return self.o.for_residual(y, ctx)
