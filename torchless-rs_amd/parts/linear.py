"""Products with a weight matrix stored [out, in] as the checkpoint has it
(out[r] = sum_c W[r,c] x[c], src/loader/parameters.rs:551-594 of the
reference).  The kernel is chosen by what the operands are, never by the
model: float32 anywhere means the plain FMA kernel (true 32-bit)."""
from __future__ import annotations

import torch

import contextlib
import contextvars

from ..kernels import ops

# whether weights loaded now may keep tiled copies: set for the extent of one load
# (`loading_with`), per thread and task, never for the process
_tiled_copies = contextvars.ContextVar("tiled_copies", default=True)


@contextlib.contextmanager
def loading_with(tiled_copies: bool):
    """Within this block `Linear(..., tiled=True)` keeps its tiled copy only if `tiled_copies`."""
    token = _tiled_copies.set(bool(tiled_copies))
    try:
        yield
    finally:
        _tiled_copies.reset(token)


class Linear:
    """A weight [N, K] resident on the device in its stored width.  With `tiled` it
    also keeps the tiled copy (`ops.tile_weights`) that the products of steps of at
    most 16 rows read instead: memory spent for the rate at which decoding streams
    the weights (a load under `loading_with(False)` makes none).  `tile_rows`: the
    copy's own order of rows, for a kernel that wants one; then only that kernel
    reads it (`own_tiles`)."""

    def __init__(self, weight: torch.Tensor, tiled: bool = False, tile_rows: torch.Tensor = None):
        assert weight.dim() == 2
        self.weight = weight.contiguous()
        self.out_features, self.in_features = self.weight.shape
        self.tiles = self.own_tiles = None
        if (tiled and _tiled_copies.get() and self.weight.is_cuda and self.weight.dtype == torch.bfloat16
                and ops.tiles_fit(self.out_features, self.in_features)):
            copy = ops.tile_weights(self.weight, tile_rows)
            if tile_rows is None:
                self.tiles = copy
            else:
                self.own_tiles = copy

    def __call__(self, a: torch.Tensor, out: torch.Tensor, accumulate: bool = False, factor=None) -> None:
        """out[M, N] (+)= a[M, K] @ W^T; out is float32.  `factor` (`ops.RowFactor`): the
        second half of the norm that made `a`, a factor per row (at most 16 rows)."""
        if factor is not None:
            ops.gemm_bf16_norm(a, self.weight, out, accumulate, factor=factor, tiles=self.tiles)
        elif self.mid(a):
            ops.gemm_mid_bf16(a, self.weight, out, 1, accumulate)
        else:
            ops.gemm(a, self.weight, out, accumulate, tiles=self.tiles)

    def own_kernels(self, n_rows: int) -> bool:
        """Does a product of `n_rows` rows launch this package's kernels only (never the BLAS
        library's, which a captured graph must not hold)?"""
        return n_rows <= ops.own_rows(self.in_features) or self.weight.dtype != torch.bfloat16

    def mid(self, a: torch.Tensor) -> bool:
        """17..`ops.own_rows(K)` rows of bfloat16: the kernels that share the activations
        through LDS."""
        return 16 < a.shape[0] <= ops.own_rows(self.in_features) and ops.bf16_gemm_ok(a, self.weight)

    def partial(self, a: torch.Tensor, ctx, name: str):
        """The product as partial sums [S, M, N] (float32) for a reader that adds
        them up, where that pays (17..MID_ROWS rows and K worth cutting); else None."""
        if not self.mid(a):
            return None
        S = ops.mid_splits(a.shape[0], self.out_features, self.in_features, ops.compute_units(a.device))
        if S == 1:
            return None
        parts = ctx.workspace.get(name, (S, a.shape[0], self.out_features), torch.float32)
        ops.gemm_mid_bf16(a, self.weight, parts, S)
        return parts

    def wide_partial(self, a: torch.Tensor, ctx, name: str):
        """The same for MID_ROWS + 1..WIDE_ROWS rows, where the sums go to the stream: whoever reads it next adds them, a norm as it
        reads or a pass of its own; and where the rotation of a prompt's q|k|v adds them.  This rule comes before `tall_partial`'s: it asks for no norm, and takes 144 to 256 rows of wide outputs and short K
        that the other, which reckons times, leaves to the library (8,192 x 4,096 at 256 rows 36 us in four slices, 48 there)."""
        M, N, K = a.shape[0], self.out_features, self.in_features
        if not (ops.MID_ROWS < M <= ops.WIDE_ROWS and ops.bf16_gemm_ok(a, self.weight)):
            return None
        S = ops.wide_splits(M, N, K, ops.compute_units(a.device))
        if S == 1:
            return None
        parts = ctx.workspace.get(name, (S, M, N), torch.float32)
        ops.gemm_wide_bf16(a, self.weight, parts, S)
        return parts

    def rotated_partial(self, a: torch.Tensor, ctx, name: str):
        """`partial`, or `wide_partial` where the rotation of a prompt's q|k|v (`ops.rope_v_tiles`) adds the sums up sooner than the library
        stores the product: K of 4,096 and more in 8 slices at most.  Product and rotation, weights from memory, in slices / by the
        library, microseconds: 6,144 x 4,096 at 130, 192, 226 and 255 rows 28.5 / 32.2, 30.0 / 39.6, 31.1 / 32.8 and 32.1 / 33.7; 6,144 x 5,120
        31.8 / 38.0 to 37.4 / 40.6; 8,192 x 4,096 30.7 / 32.2 to 37.4 / 37.8; 10,240 x 8,192 49 / 65 to 67 / 96; 4,096 x 4,096 at 130 to
        192 rows 25.7 / 26.8 to 27.1 / 38.2; not taken: 6,144 x 3,072 26.7 / 26.2 to 30.3 / 27.7, 3,072 x 4,096 in 10 26.1 / 19.9.
        Against 64 bits the sum of slices is off by 1.7e-7 of its norm where the library's product is by 4.0e-7 (K 4,096)."""
        from .base import goes_as
        parts = self.partial(a, ctx, name)
        M, N, K = a.shape[0], self.out_features, self.in_features
        if (parts is None and M > ops.MID_ROWS and K >= 4096 and goes_as(self, Linear, "__call__")
                and ops.wide_splits(M, N, K, ops.compute_units(a.device)) <= 8):
            parts = self.wide_partial(a, ctx, name)
        return parts

    def tall_partial(self, a: torch.Tensor, ctx, name: str):
        """The same for more rows than that, and for what `wide_splits` leaves (4,096 x 4,096 at 200 to 240 rows; outputs of few channels:
        1,024 x 4,096 at 226 rows 17 us with the norm, the library's 19), where a norm that adds such sums is announced as the
        stream's next reader (without one they would take a pass of their own)."""
        norm = ctx.norm_ahead
        if a.shape[0] <= ops.MID_ROWS or norm is None or not getattr(norm, "takes_pending", False) or not ops.bf16_gemm_ok(a, self.weight):
            return None
        plan = ops.tall_plan(a.shape[0], self.out_features, self.in_features, ops.compute_units(a.device), "add", True)
        if plan is None or plan.n_split == 1:
            return None
        parts = ctx.workspace.get(name, (plan.n_split, a.shape[0], self.out_features), torch.float32)
        ops.gemm_tall_bf16(a, self.weight, parts, plan)
        return parts

    def add_into(self, a: torch.Tensor, x: torch.Tensor, ctx, name: str) -> None:
        """x += a @ W^T, now or as partial sums left in `ctx.pending`."""
        from .base import flush_pending
        flush_pending(ctx, x)
        norm = ctx.norm_ahead
        form = norm.rms_form() if norm is not None and ops.norm_split_ok(a, self.weight) else None
        if (form is not None and form.size == self.out_features and form.weight is not None
                and form.weight.dtype == torch.float32):
            # the next norm's first half rides on this product
            xt = ctx.workspace.get("prenormed_y", (a.shape[0], self.out_features), torch.bfloat16)
            ssq = ctx.workspace.get(name + "_ssq", (16, -(-self.out_features // 16)), torch.float32)
            groups = ops.gemm_bf16_norm(a, self.weight, x, accumulate=True, norm_weight=form.weight, xt=xt,
                                        ssq_out=ssq, tiles=self.tiles)
            ctx.prenormed = (norm, xt, ops.RowFactor(ssq, groups, form.size, form.eps))
            return
        parts = self.partial(a, ctx, name)
        if parts is None:
            parts = self.wide_partial(a, ctx, name)
        if parts is None:
            parts = self.tall_partial(a, ctx, name)
        if parts is None:
            self(a, x, accumulate=True)
        else:
            ctx.pending = parts


def interleave_pairs(gate: torch.Tensor, up: torch.Tensor, block: int = 32) -> torch.Tensor:
    """Rows in groups of 2*block: `block` rows of gate, then the `block` rows of
    up that belong to them: the layout of the products' paired epilogue."""
    I, K = gate.shape
    g = gate.view(I // block, block, K)
    u = up.view(I // block, block, K)
    return torch.stack([g, u], dim=1).reshape(2 * I, K).contiguous()
