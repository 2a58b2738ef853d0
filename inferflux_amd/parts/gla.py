"""Gated linear attention: a recurrence per head whose state is a matrix S [d, dv] and whose decay is a vector per token.

With ``n_heads`` heads, keys and queries of ``head_dim`` channels, values of ``v_head_dim`` and a decay projected through
``decay_rank`` numbers, for a request's tokens t = 0, 1, ...:

    q = W_q h * head_dim^(-1/2),  k = W_k h,  v = W_v h,  g = W_g h
    z = W_a2 (W_a1 h) + b_a2                               (n_heads x head_dim)
    alpha = sigmoid(z) ^ (1 / tau)                         per key channel, in float
    S_t = diag(alpha_t) S_(t-1) + k_t v_t^T,  S_(-1) = 0   per head, in float
    o_t = S_t^T q_t
    out = W_o ( rmsnorm_head(o_t) * w_norm * silu(g) )     the norm over each head's v_head_dim, one weight for all heads

What a request carries from step to step is its S: one float32 row of the engine's per-request state (``StateSpec``), laid
out as the kernel of ``csrc/gla.hip`` wants it, zeroed when the request starts.  Nothing is kept per token, so the layer
owns no cache pages.  q, k, v, g and the decay's first product come from one fused projection in the activation type; the
decay's second product gives float32, and decays, S, o, the norm and the gate are float whatever the activation type.

Tensors (``tensors`` maps the roles "q", "k", "v", "g", "o", "a1", "a2", "a2_bias", "norm" to full names; by default
``<name>.q_proj.weight`` and so on, ``<name>.a2_proj.bias``, ``<name>.norm.weight``).
"""
from __future__ import annotations

from typing import Dict, Mapping, Optional

import torch

from ..kernels import ops
from .base import Mixer, MixerBinding, register_part
from .ffn import concat_weights
from .plan import ParamSpec, StateSpec


SCAN_CHUNK = 32             # rows of a chunk where long portions are cut into chunks that run side by side
SCAN_CHUNK_MIN_ROWS = 128   # ... which happens in steps that bring some request this many rows or more
BLOCKS_MIN_ROWS = 48        # ... of heads whose chunks run on the matrix cores, where this many do,
BLOCKS_FEW_MIN_ROWS, BLOCKS_FEW_REQUESTS = 24, 8          # or this many in steps of so few requests,
BLOCKS_LONG_CHUNK, BLOCKS_LONG_ROWS = 64, 2048            # and whose chunks are longer in steps of so many rows


def chunk_rows(longest: int, n_rows: int, n_requests: int, blocks: bool) -> int:
    """Rows of a chunk in a step whose longest request brings ``longest`` rows, 0: its requests are walked whole.  us walked / in chunks of 32 on the
    matrix cores, 16 and 8 heads of 64 x 128: a request of 24 rows 33 / 21, 32 / 21, of 100 122 / 23, 122 / 22; 16 of 32 44 / 42, 43 / 32, of 48 63 / 48,
    62 / 34; 64 of 24 82 / 112, 40 / 62, of 48 146 / 146, 79 / 83, of 64 192 / 150, 103 / 84; a request of 64 beside 16 of one 80 / 47, 79 / 32.  Chunks of 32 /
    64: 200 rows 25 / 34, 23 / 33, 1,000 40 / 41, 33 / 37, 4,026 of 16 requests 123 / 113, 73 / 72, 8,192 of four 212 / 167, 114 / 92."""
    if not blocks:
        return SCAN_CHUNK if longest >= SCAN_CHUNK_MIN_ROWS else 0
    if longest < (BLOCKS_FEW_MIN_ROWS if n_requests <= BLOCKS_FEW_REQUESTS else BLOCKS_MIN_ROWS):
        return 0
    return BLOCKS_LONG_CHUNK if n_rows >= BLOCKS_LONG_ROWS else SCAN_CHUNK


@register_part("mixer", "gated_linear_attention")
class GatedLinearAttention(Mixer):
    graph_safe = True          # the kernel reads the step's layout from the context's device arrays
    adds_to_stream = True

    def __init__(self, name: str, hidden_size: int, n_heads: int, head_dim: int, v_head_dim: int, decay_rank: int, tau: float,
                 norm_eps: float, init_std: float = 0.02, tensors: Optional[Mapping[str, str]] = None):
        self.name, self.hidden_size = name, int(hidden_size)
        self.n_heads, self.head_dim, self.v_head_dim = int(n_heads), int(head_dim), int(v_head_dim)
        self.decay_rank, self.tau, self.norm_eps = int(decay_rank), float(tau), float(norm_eps)
        if min(self.n_heads, self.head_dim, self.v_head_dim, self.decay_rank) <= 0 or self.tau <= 0:
            raise ValueError(f"{name}: heads, head_dim, v_head_dim, decay_rank and tau must be positive")
        ops.gla_layout(self.head_dim, self.v_head_dim)          # (refuses head sizes the kernel has no layout for)
        self.init_std = init_std
        self.names = {k: f"{name}.{k}_proj.weight" for k in ("q", "k", "v", "g", "o", "a1", "a2")}
        self.names.update({"a2_bias": f"{name}.a2_proj.bias", "norm": f"{name}.norm.weight"})
        self.names.update(tensors or {})
        self.w_in = self.w_a2 = self.w_o = self.a2_bias = self.norm_w = None

    def state_spec(self) -> StateSpec:
        return StateSpec((ops.gla_state_floats(self.n_heads, self.head_dim, self.v_head_dim),), "float32")

    def param_specs(self) -> Dict[str, ParamSpec]:
        nm, H, s = self.names, self.hidden_size, ("normal", self.init_std)
        HD, HV, r = self.n_heads * self.head_dim, self.n_heads * self.v_head_dim, self.decay_rank
        return {
            nm["q"]: ParamSpec((HD, H), s), nm["k"]: ParamSpec((HD, H), s), nm["v"]: ParamSpec((HV, H), s),
            nm["g"]: ParamSpec((HV, H), s), nm["o"]: ParamSpec((H, HV), s), nm["a1"]: ParamSpec((r, H), s),
            nm["a2"]: ParamSpec((HD, r), ("normal", 0.5)), nm["a2_bias"]: ParamSpec((HD,), ("uniform", 0.0, 6.0)),
            nm["norm"]: ParamSpec((self.v_head_dim,), ("ones",)),
        }

    def load(self, tensors: Mapping[str, torch.Tensor]) -> None:
        nm = self.names
        self.w_in = ops.prepare_linear(concat_weights([tensors[nm[p]] for p in ("q", "k", "v", "g", "a1")]))
        self.w_a2 = ops.prepare_linear(tensors[nm["a2"]])
        self.w_o = ops.prepare_linear(tensors[nm["o"]])
        self.a2_bias = tensors[nm["a2_bias"]].float().contiguous()      # float whatever the file holds
        self.norm_w = tensors[nm["norm"]]

    def accepts_scaled_rows(self, n_rows: int) -> bool:
        return ops.takes_scaled_rows(n_rows, self.w_in)

    def forward(self, h, ctx, binding: MixerBinding, sink=None):
        state, t = binding.state, ctx.timer
        if state is None:
            raise ValueError(f"{self.name}: the mixer was given no per-request state")
        HD, HV, r = self.n_heads * self.head_dim, self.n_heads * self.v_head_dim, self.decay_rank
        rows = ops.linear(h, self.w_in)                                 # [T, q | k | v | g | a1]
        cols = (0, HD, 2 * HD, 2 * HD + HV)
        a1 = rows[:, 2 * HD + 2 * HV:] if rows.shape[0] else rows.new_empty((0, r))
        if not ops.columns_on_16_bytes(a1):
            a1 = a1.contiguous()              # (``linear`` takes columns in bfloat16 on 16 bytes)
        # (steps of single tokens: the recurrence's launch forms them where it can)
        alone = 0 < ctx.n_tokens == ctx.n_requests and rows.dtype == torch.bfloat16 and ops.gla_step_takes(a1, self.w_a2.rows, self.head_dim, self.v_head_dim)
        z = (a1, self.w_a2.rows) if alone else ops.linear(a1, self.w_a2, out_dtype=torch.float32)      # the decays' logits are never rounded
        if t is not None:
            t.mark("mixer.project")
        # A prompt's portion walked token by token leaves most of the chip idle: in bfloat16 long portions are cut into
        # chunks that run side by side.  In 32-bit the walk stays in one piece, so that a token's sums do not depend on
        # where its request was cut.  (Steps of single tokens never take the chunks: a captured layout keeps its launches.)
        chunks = None
        if rows.dtype == torch.bfloat16 and ctx.n_tokens > ctx.n_requests:
            chunk = chunk_rows(int(ctx.h_q_len.max()), ctx.n_tokens, ctx.n_requests,
                               ops.gla_takes_blocks(rows, cols, z, self.a2_bias, self.head_dim, self.v_head_dim))
            if chunk:
                chunks = ctx.derived(("scan_chunks", chunk), lambda: ops.scan_chunks(ctx.h_q_start, ctx.h_q_len, chunk, ctx.device))
        y = ops.gla_scan(rows, cols, z, self.a2_bias, self.tau, self.head_dim ** -0.5, self.norm_w,
                         self.norm_eps, self.n_heads, self.head_dim, self.v_head_dim, state, 0, ctx.q_start, ctx.q_len,
                         ctx.state_slots, chunks)
        if t is not None:
            t.mark("mixer.scan")
        if sink is not None and ops.adds_into_stream(y.shape[0], self.w_o, sink.norm_weight, sink.single_tokens):
            return ops.linear_into_stream(y, self.w_o, sink.stream, sink.norm_weight, sink.eps, sink.mult)
        return ops.linear(y, self.w_o, keep_slices=sink is not None)
