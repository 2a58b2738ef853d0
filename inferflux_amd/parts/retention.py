"""Retention: linear attention with a fixed decay per head, no softmax and no denominator; a recurrence whose state is a matrix
S [d, dv] per head.

With ``n_heads`` heads, queries and keys of ``head_dim`` channels and values of ``v_head_dim``, for a request's tokens:

    q = turn(W_q h),  k = turn(W_k h) * head_dim^(-1/2),  v = W_v h,  g = W_g h       (turn: the position part's rotation)
    S_t = decay S_(t-1) + k v^T,  S_(-1) = 0;  o_t = S_t^T q                          decay: one number per head
    out = W_o ( rms(o_t) silu(g) )                           each head's o over its root mean square, no weight

What a request carries from step to step is S: one float32 row of the engine's per-request state (``StateSpec``), laid out as
the kernels of ``csrc/retention.hip`` want it, zeroed when the request starts.  Nothing is kept per token, so the layer owns no
cache pages.  q, k, v and g come from one fused projection (in float for steps of few rows, else in the activation type);
everything behind it is float.

Tensors (``tensors`` maps the roles "q", "k", "v", "g", "o" to full names; by default ``<name>.q_proj.weight`` and so on).
"""
from __future__ import annotations

import math
from typing import Dict, Mapping, Optional, Sequence

import torch

from ..kernels import ops
from .base import Mixer, MixerBinding, build_part, register_part
from .ffn import concat_weights
from .plan import ParamSpec, PartSpec, StateSpec


CHUNK_MIN_ROWS = 64         # a step that brings some request this many rows or more takes the chunks
LOG2_OF_ZERO = -3.0e38      # (finite: a decay of 0 to the power 0 is 1)


@register_part("mixer", "retention")
class Retention(Mixer):
    graph_safe = True          # every kernel reads the step's layout from the context's device arrays
    adds_to_stream = True

    def __init__(self, name: str, hidden_size: int, n_heads: int, head_dim: int, v_head_dim: int, decay: Sequence[float], norm_eps: float,
                 position: PartSpec, init_std: float = 0.02, tensors: Optional[Mapping[str, str]] = None):
        self.name, self.hidden_size = name, int(hidden_size)
        self.n_heads, self.head_dim, self.v_head_dim = int(n_heads), int(head_dim), int(v_head_dim)
        self.decay, self.norm_eps, self.init_std = tuple(float(x) for x in decay), float(norm_eps), init_std
        if min(self.n_heads, self.head_dim, self.v_head_dim) <= 0 or len(self.decay) != self.n_heads:
            raise ValueError(f"{name}: {n_heads} heads of {head_dim} x {v_head_dim} with {len(self.decay)} decays")
        if not all(0.0 <= x <= 1.0 for x in self.decay):
            raise ValueError(f"{name}: decays between 0 and 1, got {self.decay}")
        ops.retention_layout(self.head_dim, self.v_head_dim)          # (refuses head sizes the kernel has no layout for)
        self.position = build_part("position", position)
        if self.position.needs_apply or getattr(self.position, "style", "split_half") != "split_half":
            raise ValueError(f"{name}: retention needs a position part that gives the kernels a table of split-half rotations")
        self.names = {k: f"{name}.{k}_proj.weight" for k in ("q", "k", "v", "g", "o")}
        self.names.update(tensors or {})
        self.qk_width, self.v_width = self.n_heads * self.head_dim, self.n_heads * self.v_head_dim
        self.w_in = self.w_o = self.decay_t = self.log2_decay = None

    def state_spec(self) -> StateSpec:
        return StateSpec((ops.retention_state_floats(self.n_heads, self.head_dim, self.v_head_dim),), "float32")

    def param_specs(self) -> Dict[str, ParamSpec]:
        nm, H, s, QK, V = self.names, self.hidden_size, ("normal", self.init_std), self.qk_width, self.v_width
        return {nm["q"]: ParamSpec((QK, H), s), nm["k"]: ParamSpec((QK, H), s), nm["v"]: ParamSpec((V, H), s),
                nm["g"]: ParamSpec((V, H), s), nm["o"]: ParamSpec((H, V), s)}

    def load(self, tensors: Mapping[str, torch.Tensor]) -> None:
        nm = self.names
        self.w_in = ops.prepare_linear(concat_weights([tensors[nm[p]] for p in ("q", "k", "v", "g")]))
        self.w_o = ops.prepare_linear(tensors[nm["o"]])
        device = self.w_in.rows.device
        self.decay_t = torch.tensor(self.decay, dtype=torch.float32, device=device)
        self.log2_decay = torch.tensor([math.log2(x) if x > 0 else LOG2_OF_ZERO for x in self.decay], dtype=torch.float32, device=device)

    def accepts_scaled_rows(self, n_rows: int) -> bool:
        return ops.takes_scaled_rows(n_rows, self.w_in)

    def forward(self, h, ctx, binding: MixerBinding, sink=None):
        state, t = binding.state, ctx.timer
        if state is None:
            raise ValueError(f"{self.name}: the mixer was given no per-request state")
        QK, V, dtype = self.qk_width, self.v_width, h.dtype
        _, rot_dims, cos, sin = self.position.kernel_args(ctx)
        # A prompt's portion walked token by token leaves most of the chip idle: in bfloat16 long portions are cut into chunks
        # that run side by side.  In 32-bit the walk stays in one piece, so that a token's sums do not depend on where its
        # request was cut.  (Steps of single tokens never take the chunks: a captured layout keeps its launches.)
        single = ctx.n_tokens == ctx.n_requests
        chunks = None
        if not single and ops.retention_takes_chunks(dtype, self.head_dim, self.v_head_dim) and int(ctx.h_q_len.max()) >= CHUNK_MIN_ROWS:
            chunks = ctx.derived(("scan_chunks", ops.RETENTION_CHUNK),
                                 lambda: ops.scan_chunks(ctx.h_q_start, ctx.h_q_len, ops.RETENTION_CHUNK, ctx.device))
        # few rows: one product whose float sums are read as they are; many: the activation type for what is wide
        wide = chunks is None and ops.streams_weight(h.shape[0], self.w_in)
        rows = ops.linear(h, self.w_in, out_dtype=torch.float32) if wide else ops.linear(h, self.w_in)
        if t is not None:
            t.mark("mixer.project")
        y = ops.retention(rows, (0, QK, 2 * QK, 2 * QK + V), cos, sin, rot_dims, self.decay_t, self.log2_decay, self.norm_eps, self.n_heads,
                          self.head_dim, self.v_head_dim, state, ctx.q_start, ctx.q_len, ctx.state_slots, dtype, single, chunks)
        if t is not None:
            t.mark("mixer.scan")
        if sink is not None and ops.adds_into_stream(y.shape[0], self.w_o, sink.norm_weight, sink.single_tokens):
            return ops.linear_into_stream(y, self.w_o, sink.stream, sink.norm_weight, sink.eps, sink.mult)
        return ops.linear(y, self.w_o, keep_slices=sink is not None)
