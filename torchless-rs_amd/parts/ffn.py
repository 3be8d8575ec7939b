"""Gated feed-forward: down( act(gate y) * (up y) ).  With act = silu,
silu(g) = g / (1 + e^-g), it is SwiGLU (src/model/modules/mlp.rs:23-45,
src/kernels/mod.rs:546-548 of the reference); `activation` chooses another
function of the gate (`ops.ACTIVATIONS`: gelu_tanh, the tanh form of gelu;
swish_clamped, g' logistic(alpha g') (u' + shift) on a gate clamped from above and
an up clamped on both sides, whose constants come in `activation_constants`).
gate and up are bound under their own names (`names`: the leaf names are
parameters, and a checkpoint that stores gate|up as one tensor binds that one)
and laid side by side at load so that one product serves both."""
from __future__ import annotations

from typing import Dict, Optional

import torch

from ..kernels import ops
from ..weights.binding import WeightSpec
from .base import FeedForward, goes_as, register_part, take_row_factor, take_row_norm
from .linear import Linear, interleave_pairs


class SwiGLU(FeedForward):
    graph_safe = True
    row_wise = True
    closes_stream = True          # its last write to the stream is `Linear.add_into`
    takes_row_factor = True       # its gate|up product can do the division of the norm before it

    # leaf names of the tensors under `prefix`; "gate_up": one tensor [gate | up] by rows instead of the two
    NAMES = {"gate": "gate_proj.weight", "up": "up_proj.weight", "down": "down_proj.weight", "gate_up": None}

    def __init__(self, hidden_size: int, intermediate_size: int, prefix: str = "mlp.",
                 names: Optional[Dict[str, Optional[str]]] = None, activation: str = "silu",
                 activation_constants: Optional[Dict[str, float]] = None):
        if activation not in ops.ACTIVATIONS:
            raise ValueError(f"gated feed-forward: no activation {activation!r}; there are {sorted(ops.ACTIVATIONS)}")
        need = set(ops.ACTIVATION_CONSTANTS.get(activation, ()))
        if set(activation_constants or {}) != need:
            raise ValueError(f"gated feed-forward: {activation!r} takes the constants {sorted(need)}, "
                             f"got {sorted(activation_constants or {})}")
        self.activation = activation
        self.constants = dict(activation_constants or {}) or None
        self.pair = (activation, self.constants) if self.constants else activation     # as the products' epilogue takes it
        self.H = int(hidden_size)
        self.I = int(intermediate_size)
        self.prefix = prefix
        unknown = set(names or {}) - set(self.NAMES)
        if unknown:
            raise ValueError(f"swiglu: no tensors called {sorted(unknown)}; there are {sorted(self.NAMES)}")
        self.names = dict(self.NAMES, **(names or {}))
        self.gate_up = None
        self.down = None

    def may_capture(self, n_rows: int) -> bool:
        return self.gate_up is not None and self.gate_up.own_kernels(n_rows) and self.down.own_kernels(n_rows)

    def weight_specs(self) -> Dict[str, WeightSpec]:
        p, nm = self.prefix, self.names
        if nm["gate_up"]:
            return {p + nm["gate_up"]: WeightSpec((2 * self.I, self.H)), p + nm["down"]: WeightSpec((self.H, self.I))}
        return {p + nm["gate"]: WeightSpec((self.I, self.H)),
                p + nm["up"]: WeightSpec((self.I, self.H)),
                p + nm["down"]: WeightSpec((self.H, self.I))}

    def load(self, tensors, compute_dtype) -> None:
        p, nm = self.prefix, self.names
        if nm["gate_up"]:
            g, u = tensors[p + nm["gate_up"]][:self.I], tensors[p + nm["gate_up"]][self.I:]
        else:
            g, u = tensors[p + nm["gate"]], tensors[p + nm["up"]]
        if g.dtype != u.dtype:
            g, u = g.to(torch.float32), u.to(torch.float32)
        # bfloat16 on the matrix cores: gate and up rows interleaved so that the product's
        # epilogue applies silu(gate) * up itself and writes bfloat16
        self.paired = (compute_dtype == torch.bfloat16 and g.dtype == torch.bfloat16 and self.I % 32 == 0
                       and self.H % 8 == 0 and self.activation in ops.PAIR_EPILOGUES)
        self.gate_up = Linear(interleave_pairs(g, u) if self.paired else torch.cat([g, u], dim=0))
        self.down = Linear(tensors[p + nm["down"]], tiled=True)

    def norms_rows(self, ctx, norm, x: torch.Tensor, run) -> bool:
        return (goes_as(self, SwiGLU, "forward", "_hidden") and ctx.dtype == torch.float32 and self._around(x)
                and ops.row_norm_ok(norm.rms_form(), self.H))

    def _around(self, y: torch.Tensor) -> bool:
        """Does the 32-bit path do the product and the activation in one launch?  (Not for a weight with a product of its own.)"""
        return self.I % 4 == 0 and type(self.gate_up) is Linear and ops.plain_around_ok(y, self.gate_up.weight)

    def forward(self, ctx, y: torch.Tensor, x: torch.Tensor) -> None:
        self.down.add_into(self._hidden(ctx, y), x, ctx, "ffn_down_parts")

    def produce(self, ctx, y: torch.Tensor, out: torch.Tensor) -> None:
        """The result stored in `out` (float32 [n, H]) instead of added to the stream."""
        self.down(self._hidden(ctx, y), out)

    def _hidden(self, ctx, y: torch.Tensor) -> torch.Tensor:
        n = y.shape[0]
        h = ctx.workspace.get("ffn_h", (n, self.I), ctx.dtype)
        factor = take_row_factor(ctx, usable=self.paired and ops.norm_split_ok(y, self.gate_up.weight))
        if factor is not None:
            ops.gemm_bf16_norm(y, self.gate_up.weight, h, silu_pair=True, factor=factor, pair_act=self.pair)
        elif self.paired and self.gate_up.mid(y):
            ops.gemm_mid_bf16(y, self.gate_up.weight, h, 1, silu_pair=True, pair_act=self.pair)
        elif self.paired and ops.bf16_gemm_ok(y, self.gate_up.weight):
            plan = ops.tall_plan(n, 2 * self.I, self.H, ops.compute_units(y.device), "pair")
            if plan is not None and h.data_ptr() % 16 == 0:
                ops.gemm_tall_bf16(y, self.gate_up.weight, h, plan, silu_pair=True, pair_act=self.pair)
            elif n > ops.LIBRARY_ROWS:
                gu = ctx.workspace.get("ffn_gu16", (n, 2 * self.I), torch.bfloat16)
                ops.gemm_library(y, self.gate_up.weight, gu)
                ops.silu_mul_pairs(gu, h, self.activation, self.constants)
            else:
                ops.gemm_bf16(y, self.gate_up.weight, h, silu_pair=True, pair_act=self.pair)
        elif h.dtype == torch.float32 and self._around(y):       # norm, product and activation in one
            ops.gemm_plain_pair(y, self.gate_up.weight, h, self.activation, self.constants, norm=take_row_norm(ctx))
        else:
            gu = ctx.workspace.get("ffn_gu", (n, 2 * self.I), torch.float32)
            self.gate_up(y, gu)
            ops.act_mul(gu, h, self.activation, self.constants)
        return h


register_part("ffn", "swiglu", SwiGLU)
register_part("ffn", "gated", SwiGLU)          # the same part under the name that fits any activation
