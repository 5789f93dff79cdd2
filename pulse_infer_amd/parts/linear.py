"""y = x W^T for a weight stored [out, in] (reference: src/layer/linear.cpp:213).

Four products stand behind it:

* few rows (decoding, short portions) of bfloat16: this package's weight-streaming
  matrix-core kernel, which can also add into the float32 residual or apply SwiGLU;
* 65 rows and more of bfloat16: this package's product with several stages of its
  operands on their way through LDS, which can apply SwiGLU on the way out or leave
  float32 results of shares of the inner dimension (``takes_stages`` and
  ``stage_shares_for`` say where it is the faster one);
* else the vendor library's product (torch.matmul / torch.mm, i.e. hipBLASLt/rocBLAS,
  float32 accumulation, bfloat16 or float32 output), as the reference uses cuBLAS
  (src/ops/kernels/cuda/matmul_kernel.cu:132-154); ``OWN_MANY_ROWS`` says which
  products of many rows go where;
* the float32 run, and any weight kept in 32-bit: this package's own kernel on the
  float32 matrix instruction, with no reduced-precision mode anywhere.
"""
from __future__ import annotations

import os
from typing import Any, Optional

import torch

from ..ops import kernels, timing
from ..ops.device import compute_units
from .base import LazyNorm, RowStats, Workspace


# Which products of many rows (256 and more) run as this package's instead of the library's: "stages", the product in
# stages where it is the faster one (``takes_stages``); or the same in tiles of 256 x 256 throughout, "swiglu": for gate and up with
# SwiGLU inside (the others as with "stages"), "all": for every product of bfloat16 (a step then makes no library call); "none": none of
# them.  (Products of fewer rows are not its business: 65 to 255
# of them run in stages, where that is the faster one, whatever it says.)  PULSE_OWN_PRODUCTS sets it.
# Measured, prompts of the 8B shape: 509 tokens 8.7 ms with "stages", 11.3 with "none" (whose updates in shares are made one
# after the other, see ``add_into``); 2,048 tokens 24.9 with "stages", 26.9 with "none"; 8,192 106.5 and 108.8.
OWN_MANY_ROWS = os.environ.get("PULSE_OWN_PRODUCTS", "stages")
if OWN_MANY_ROWS not in ("none", "stages", "swiglu", "all"):
    raise ValueError(f"PULSE_OWN_PRODUCTS must be none, stages, swiglu or all, not '{OWN_MANY_ROWS}'")
library_calls = 0   # products that went to the vendor library so far (a step that made none can be recorded as a graph)


class Linear:
    def __init__(self, weight: torch.Tensor, mode: str):
        if weight.dim() != 2:
            raise ValueError(f"a linear weight must be a matrix, got shape {tuple(weight.shape)}")
        self.weight = weight
        self.out_features, self.in_features = weight.shape
        self.mode = mode
        self.library = mode == "bfloat16" and weight.dtype == torch.bfloat16

    def takes_lazy(self, x: LazyNorm, rows: Optional[int] = None) -> bool:
        """Whether the product can take rows that have not been normalised yet and scale its result instead."""
        n = self.out_features if rows is None else rows
        return (self.library and kernels.gemm_skinny_fusable(x.shape[0], n, self.in_features)
                and x.x.dtype == torch.bfloat16 and kernels.gemm_skinny_ok(x.x, self.weight))

    def forward(self, x, out: torch.Tensor, rows: Optional[int] = None, swiglu: Any = False,
                own: bool = True) -> torch.Tensor:
        """``out`` [M, out_features] receives the product; its storage type is bfloat16 or float32.  ``x`` may be a
        ``LazyNorm`` that ``takes_lazy`` accepted.  ``swiglu``: few rows of a slab-interleaved gate/up weight only.
        ``own=False``: 17 to 64 rows go to the library although this package has a product for them (a caller that
        measured the library faster for its shape)."""
        w = self.weight if rows is None else self.weight[:rows]
        if isinstance(x, LazyNorm):
            kernels.gemm_skinny(x.x, w, out, swiglu=swiglu, row_scale=(x.sumsq, x.eps))
            return out
        if swiglu:   # (True, or the gate's activation by name where it is not silu; the tiled product knows silu)
            if x.shape[0] > self.MID_ROWS[1]:
                if kernels.gate_code(swiglu) != 1:
                    raise ValueError("the tiled product applies silu only")
                if self.takes_stages(x, w, swiglu=True):
                    kernels.gemm_stages(x, w, out, swiglu=True)
                else:
                    kernels.gemm_tile(x, w, out, swiglu=True)
            elif x.shape[0] > kernels.SKINNY_FAST_ROWS:
                kernels.gemm_mid(x, w, out, swiglu=swiglu, waves=self.swiglu_waves_for(x.shape[0]) or 4)
            else:
                kernels.gemm_skinny(x, w, out, swiglu=swiglu)
            return out
        if self.library and x.dtype == torch.bfloat16:
            few = x.shape[0] <= kernels.SKINNY_FAST_ROWS
            if few and kernels.gemm_skinny_ok(x, w):
                kernels.gemm_skinny(x, w, out)
                return out
            if own and self.takes_own_rows(x, w, out):
                # 17 to 64 rows: X through LDS, 16 weight rows a wavefront.  A float32 result (logits) is the "parts"
                # output with one share; many weight rows take wide workgroups, few take narrow ones so that there
                # are enough of them (measured: logits of a 152K vocabulary 212 to 237 us against the library's 276 to
                # 281; 6,144 rows of qkv 17 to 21 us against 15 to 18, which a step without a library call, recorded
                # and replayed as a whole, makes up several times over).
                if self.takes_shared_k(x, w, out):
                    # few weight rows (qkv): a workgroup owns two 16-row slabs and all of K, which its wavefronts
                    # share out among themselves (6,144 weight rows of 4,096: 14.1 / 15.0 / 18.7 us at 24 / 32 / 64
                    # rows against 17.2 / 17.1 / 22.2 with a wavefront a slab; the library 14.7 / 15.1 / 17.8)
                    kernels.gemm_rows(x, w, out, slabs=2)
                    return out
                waves = 10 if w.shape[0] >= 64 * compute_units() else 2
                kernels.gemm_mid(x, w, out.view(1, *out.shape) if out.dtype == torch.float32 else out, waves=waves)
                return out
            if own and out.dtype == torch.bfloat16 and self.takes_stages(x, w) and out.stride(1) == 1 \
                    and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0:
                kernels.gemm_stages(x, w, out)
                return out
            if own and out.dtype == torch.float32 and out.is_contiguous() and self.takes_stages_float32(x, w) \
                    and out.data_ptr() % 16 == 0:
                kernels.gemm_stages(x, w, out.view(1, *out.shape))
                return out
            if own and out.dtype == torch.bfloat16 and self.takes_tiles(x, w) and out.stride(1) == 1 \
                    and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0:
                kernels.gemm_tile(x, w, out)
                return out
            if not self.rows_aligned(x, w):
                # The vendor library is handed only operands whose rows keep 16-byte alignment (inner sizes that are
                # multiples of 8, which every shape of a real model is); anything else goes through this package's
                # float32 product, which takes any shape and guards every access.
                kernels.gemm_f32(x, w, out)
                return out
            global library_calls
            library_calls += 1
            if out.dtype == torch.bfloat16:
                with timing.region("library matmul"):
                    torch.matmul(x, w.t(), out=out)
                return out
            if out.dtype == torch.float32 and out.is_contiguous():
                # float32 results of many rows: the library's product with a float32 output
                with timing.region("library matmul (float32 out)"):
                    torch.mm(x, w.t(), out_dtype=torch.float32, out=out)
                return out
            if w.shape[1] % 8 == 0:  # otherwise the few-rows kernel, 64 rows at a time
                for r0 in range(0, x.shape[0], kernels.SKINNY_MAX_ROWS):
                    kernels.gemm_skinny(x[r0:r0 + kernels.SKINNY_MAX_ROWS], w, out[r0:r0 + kernels.SKINNY_MAX_ROWS])
                return out
        kernels.gemm_f32(x, w, out)
        return out

    def add_into(self, x: torch.Tensor, residual: torch.Tensor, scratch: torch.Tensor,
                 workspace: Optional[Workspace] = None, next_scale: Optional[torch.Tensor] = None,
                 next_offset: float = 0.0, leave_stats: bool = True):
        """residual += x W^T, in one of six ways.  Few rows: the kernel adds into the residual itself and None is
        returned, or, given a workspace and a shape the fused kernel takes, the ``RowStats`` of the updated rows (their
        sums of squares and a rounded copy, multiplied column by column by ``next_scale``, the weight of the norm that
        reads the residual next, ``next_offset`` added to each in float32: with these the next product can do without a
        norm kernel before it).  17 to
        192 rows, given a workspace: the product's inner dimension is shared out over workgroups and the shares' float32
        results [parts, rows, out] are returned as the update, which the next norm adds up in order; 65 to 512 rows of a
        weight that is not small, and more rows of a product with a wide inner dimension and a narrow output: the same from
        the product in stages (``stage_shares_for``), from the tiled one if all products are to be it, or from the library's
        if none of them is to be this package's.
        Otherwise the product is written to ``scratch`` and returned for the caller to add.  ``leave_stats=False``:
        no ``RowStats`` are made (their buffers are the workspace's, one set a width: a caller that still reads the
        set of the rows as they were before this update says so)."""
        splits = self.stage_shares_for(x) if workspace is not None else 0
        if splits:
            rows = x.shape[0]
            parts = workspace.buffer(f"linear.parts.{self.out_features}.{self.in_features}", splits * rows,
                                     self.out_features, torch.float32).view(splits, rows, self.out_features)
            kernels.gemm_stages(x, self.weight, parts)
            return parts
        splits, waves = self.shares_and_waves_for(x) if workspace is not None else (0, 0)
        if splits:
            rows = x.shape[0]
            parts = workspace.buffer(f"linear.parts.{self.out_features}.{self.in_features}", splits * rows,
                                     self.out_features, torch.float32).view(splits, rows, self.out_features)
            kernels.gemm_mid(x, self.weight, parts, splits=splits, waves=waves)
            return parts
        splits = self.tile_shares_for(x) if workspace is not None else 0
        if splits:
            rows = x.shape[0]
            parts = workspace.buffer(f"linear.parts.{self.out_features}.{self.in_features}", splits * rows,
                                     self.out_features, torch.float32).view(splits, rows, self.out_features)
            kernels.gemm_tile(x, self.weight, parts)
            return parts
        splits = self.library_shares_for(x) if workspace is not None and self.operands_ok(x) else 0
        if splits:
            # Many rows but few output tiles (down: a wide inner dimension, a narrow output) that the product in stages is
            # not to take: the library's product, a share of the inner dimension after the other, with float32 results
            # that the next norm adds up in order.  (Not as one batched product: its right operand would be a transposed
            # view of bfloat16, a form that is unsafe on this stack, and a copy of the weight costs more than it gains.)
            rows, share = x.shape[0], self.in_features // splits
            parts = workspace.buffer(f"linear.parts.{self.out_features}.{self.in_features}", splits * rows,
                                     self.out_features, torch.float32).view(splits, rows, self.out_features)
            global library_calls
            library_calls += 1
            with timing.region("library matmul in shares"):
                for s in range(splits):
                    cut = slice(s * share, (s + 1) * share)
                    torch.mm(x[:, cut], self.weight[:, cut].t(), out_dtype=torch.float32, out=parts[s])
            return parts
        if (self.library and x.dtype == torch.bfloat16 and x.shape[0] <= kernels.SKINNY_FAST_ROWS
                and kernels.gemm_skinny_ok(x, self.weight)):
            if (workspace is not None and leave_stats
                    and kernels.gemm_skinny_fusable(x.shape[0], self.out_features, self.in_features)):
                sums = workspace.buffer(f"linear.sumsq.{self.out_features}", x.shape[0], (self.out_features + 15) // 16,
                                        torch.float32)
                rounded = workspace.buffer(f"linear.rounded.{self.out_features}", x.shape[0], self.out_features,
                                           torch.bfloat16)
                scaled = next_scale is not None and next_scale.dtype == torch.bfloat16 \
                    and next_scale.numel() == self.out_features and next_scale.is_contiguous()
                kernels.gemm_skinny(x, self.weight, residual, add=True, sumsq_out=sums, copy_out=rounded,
                                    copy_scale=next_scale if scaled else None,
                                    copy_offset=next_offset if scaled else 0.0)
                return RowStats(sums, rounded, next_scale if scaled else None, next_offset if scaled else 0.0)
            kernels.gemm_skinny(x, self.weight, residual, add=True)
            return None
        return self.forward(x, scratch)

    MID_ROWS = (17, 64)          # where the product with X shared through LDS and SwiGLU inside beats the library's
                                 # product followed by the SwiGLU kernel
    SHARES_ROWS = (17, 192)      # where a product that adds into the residual has its inner dimension shared out over
                                 # workgroups, from 65 rows on if the product in stages does not take it (measured on the 8B shape: 1% of a decoding step at 17 to 32 rows, 4% at
                                 # 48, 6% at 64; at 96 to 192 rows the library takes 22 to 33 us for o and 55 to 90 us
                                 # for down, the shared-out product 16 to 22 and 33 to 47.  Up to 16 rows the few-rows
                                 # kernel stands: it leaves what the next product needs to do without a norm kernel,
                                 # and a step of 13 rows is 3% faster with it, one of 16 rows as fast)

    LIBRARY_SHARES_MIN_K = 8192  # inner dimensions from here on are worth sharing out beyond 192 rows
    LIBRARY_TILE = 256           # the library's output tiles are about this large in both directions

    def library_shares_for(self, x: torch.Tensor) -> int:
        """Whether an update of more than 192 rows has so few output tiles and so wide an inner dimension that it is to be
        made in shares beyond the sizes that go in stages anyway, and into how many the library's is cut (``OWN_MANY_ROWS``
        "none"); 0: not at all.  Measured (8B, 14B and 32B shapes of down, 272 to 2,048 rows): up to about 100 tiles shares
        win (14B shape at 544 rows 179 -> 102 us with the library's products side by side, 84 in stages); in stages also while two
        shares fill the chip once, half as many tiles as compute units (us, shares with their cost in the next norm / the library's:
        4,096 x 12,288 at 2,048 rows 150 / 175, 5,120 x 17,408 at 1,536 203 / 349, 2,560 x 9,728 at 3,000 116 / 133; beyond, 5,120 x
        17,408 at 2,048 303 / 273, 5,120 x 8,192 159 / 134).  Products with an inner dimension of 4,096 to 8,192 (o) gain 5 us at most."""
        rows = x.shape[0]
        if not (self.library and x.dtype == torch.bfloat16 and rows > self.SHARES_ROWS[1]
                and self.in_features >= self.LIBRARY_SHARES_MIN_K and x.is_contiguous()
                and self.weight.is_contiguous() and self.out_features % 4 == 0):
            return 0
        tile = self.LIBRARY_TILE
        tiles = ((rows + tile - 1) // tile) * ((self.out_features + tile - 1) // tile)
        splits = 4 if tiles <= 50 else (2 if tiles <= (100 if OWN_MANY_ROWS == "none" else compute_units() // 2) else 0)
        while splits > 1 and (self.in_features % splits or (self.in_features // splits) % 64):
            splits //= 2
        return splits if splits > 1 else 0

    @staticmethod
    def rows_aligned(x: torch.Tensor, w: torch.Tensor) -> bool:
        """Whether the rows of both bfloat16 operands start at multiples of 16 bytes."""
        return (x.shape[1] % 8 == 0 and (x.shape[0] <= 1 or x.stride(0) % 8 == 0)
                and (w.shape[0] <= 1 or w.stride(0) % 8 == 0) and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)

    def operands_ok(self, x: torch.Tensor) -> bool:
        """Contiguous, aligned bfloat16 rows of a length the kernels' 16-byte loads take."""
        w = self.weight
        return (x.dim() == 2 and x.shape[1] % 8 == 0 and x.stride(1) == 1 and w.stride(1) == 1
                and (x.shape[0] <= 1 or x.stride(0) % 8 == 0) and (w.shape[0] <= 1 or w.stride(0) % 8 == 0)
                and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0)

    def takes_own_rows(self, x: torch.Tensor, w: torch.Tensor, out: torch.Tensor) -> bool:
        """Whether a plain product of this many rows (bfloat16 or float32 result) runs as this package's product for
        17 to 64 rows instead of the library's."""
        rows = x.shape[0]
        if not (self.MID_ROWS[0] <= rows <= self.MID_ROWS[1] and self.operands_ok(x) and w.stride(1) == 1
                and kernels.gemm_mid_takes(rows, w.shape[0], w.shape[1])):
            return False
        if out.dtype == torch.float32:
            return out.is_contiguous() and out.data_ptr() % 16 == 0 and w.shape[0] % 4 == 0
        return out.dtype == torch.bfloat16 and out.stride(1) == 1 and out.stride(0) % 4 == 0 and out.data_ptr() % 16 == 0

    # Where the product in stages is the fastest (more figures are beside its kernel).  With SwiGLU inside: wherever it takes the
    # shape (us against the library's product and the pass behind it: 24,576 x 4,096 at 357 / 512 / 800 / 2,048 / 8,192 rows 62 / 80 /
    # 147 / 284 / 1,116 against 91 / 104 / 165 / 337 / 1,305; 34,816 x 5,120 at 544 / 2,048 183 / 549 against 218 / 664; 51,200 x 5,120 at
    # 300 / 640 / 4,096 185 / 318 / 1,472 against 203 / 359 / 1,880; 19,456 x 2,560 at 257 / 3,000 40 / 231 against 54 / 290; over 240 sizes of
    # 16 weights from 2,048 x 2,048 and 4,096 x 1,024 on 0.72 of their time, the worst 9,728 x 2,560 and 16,384 x 3,072 at 257 rows 1.06 and
    # 1.09, 2,048 x 8,192 at 1,536 and 3,000 1.14 and 1.07).  Plain products: see ``fills_stages``.  Updates in shares: up to 512 rows all that are not small (4,096 x 4,096 at 512 rows 25 us against
    # the library's 28, 2,560 x 9,728 at 357 28 against 40), beyond those of a wide inner dimension and few tiles
    # (``library_shares_for``).  Small products stay where they are.
    STAGE_ROWS = (65, 256)              # in shares any of these (the last one if ``OWN_MANY_ROWS`` leaves it to it); with SwiGLU from the first on
    STAGE_ROWS_SHARES = 512             # beyond, only where ``library_shares_for`` says so
    STAGE_CUT_ROWS = 128                # the rows that updates of up to 192 rows are cut into shares for
    STAGE_RATE = 925                    # plain products of more rows: estimated flops a picosecond
    STAGE_LONG_K = (12288, 16384)       # and inner dimensions, see ``fills_stages``
    STAGE_SHORT_K = 512
    STAGE_MIN_WEIGHT = 1 << 22
    STAGE_FAR = 1 << 23                 # values between rows: what lies further apart goes in small tiles, which the estimate does not know of

    def takes_stages(self, x: torch.Tensor, w: Optional[torch.Tensor] = None, swiglu: bool = False) -> bool:
        """Whether a bfloat16 product of this many rows (with SwiGLU inside, or as it is) runs as this package's product
        in stages."""
        w = self.weight if w is None else w
        return self.may_stage(x, w, swiglu) and (swiglu or self.fills_stages(x.shape[0], *w.shape))

    def may_stage(self, x: torch.Tensor, w: torch.Tensor, swiglu: bool = False) -> bool:
        """Whether the product in stages takes these operands, ``OWN_MANY_ROWS`` allowing."""
        rows, (n, k) = x.shape[0], w.shape
        if not (self.library and x.dtype == torch.bfloat16 and self.STAGE_ROWS[0] <= rows
                and n * k >= self.STAGE_MIN_WEIGHT and self.operands_ok(x) and kernels.gemm_stages_takes(rows, n, k, swiglu)):
            return False
        if rows > self.STAGE_ROWS_SHARES and max(x.stride(0), w.stride(0)) >= self.STAGE_FAR:
            return False
        return rows < self.TILE_MIN_ROWS or (OWN_MANY_ROWS != "none" and not self.takes_tiles(x, w, swiglu))

    STAGE_RATE_FLOAT32 = 1000           # with float32 results, which take twice as long to store

    def takes_stages_float32(self, x: torch.Tensor, w: torch.Tensor) -> bool:
        """Whether a product of more than ``STAGE_ROWS_SHARES`` rows with float32 results runs as this package's product in stages:
        by its estimate (us, library / this, by estimated flops a picosecond: 5,120 x 5,120 at 1,024 rows (672) 53 /
        62, 8,192 x 2,048 at 1,024 (922) 33 / 38; 5,120 x 5,120 at 1,536 (1,008) 75 / 71, 4,096 x 8,192 at 2,048 (1,075) 112 /
        110, 32,000 x 4,096 at 544 (1,116) 142 / 128, 12,288 x 4,096 at 800 (1,080) 70 / 75 and 4,096 (1,498) 306 / 283, 8,192 x 2,048 at
        4,096 (1,498) 118 / 113; from 1,000 on 0.93 of the library's time over the 51 sizes measured, one of them more than 3 % slower)."""
        rows, (n, k) = x.shape[0], w.shape
        return (rows > self.STAGE_ROWS_SHARES and self.may_stage(x, w)
                and kernels.gemm_stages_time(rows, n, k) * 1000 * self.STAGE_RATE_FLOAT32 <= 2 * rows * n * k)

    def fills_stages(self, rows: int, n: int, k: int) -> bool:
        """Whether a plain product's tiles keep enough compute units busy: its inner dimension cannot be cut (the result is
        bfloat16), as the library's can, so it is the slower one where most units have no tile.

        Measured over 28 weights of 576 to 65,536 rows and 1,024 to 8,192 columns (tiles a unit and round: us, library / this):
        576 x 8,192 at 128 rows (0.07) 14 / 36, 1,536 x 7,168 at 97 (0.19) 19 / 28, 2,048 x 4,096 at 128 (0.25) 12.5 / 20,
        4,096 x 4,096 at 97 (0.50) 16 / 18, 10,240 x 5,120 at 97 (0.62) 34 / 39; 6,144 x 4,096 at 97 (0.75) 23 / 19, 4,096 x 4,096
        at 160 (0.75) 27 / 19, 7,168 x 4,096 at 192 (0.88) 35 / 28, 8,192 x 2,048 at 224 (1.0) 24 / 17; of 2,048 columns and
        fewer already 3,072 x 2,048 at 97 (0.38) 12 / 11, 4,096 x 1,024 at 65 (0.50) 11 / 7.  Beyond 256 rows the library's own
        tiles fill: 8,192 x 8,192 at 333 (0.75) 66 / 75, 6,144 x 2,560 at 300 (0.94) 22 / 24, but 6,144 x 4,096 at 357 (0.75, tiles
        of 96 x 128) 36 / 32, 8,192 x 2,048 at 300 (0.75) 24 / 21, 6,144 x 4,096 at 512 (1.0) 37 / 34.

        Beyond 512 rows its estimate decides, that is how far its tiles fill their rounds and how large they are (estimated flops a
        picosecond: us, library / this): 1,024 x 4,096 at 8,192 (922) 57 / 66, 8,192 x 4,096 at 1,024 (922) 59 / 66, 10,240 x 5,120 at 544
        (714) 64 / 69; 6,144 x 4,096 at 1,200 (945) 57 / 57, 1,536 (1,210) 70 / 59 and 2,048 (1,383) 81 / 74, 5,120 x 5,120 at 1,536 (1,008)
        76 / 70 and 8,192 (1,337) 454 / 309, 10,240 x 5,120 at 1,200 (1,097) 128 / 107, 4,096 x 4,096 at 2,048 (1,075) 59 / 57.  Two kinds
        of products stay with the library all the same.  Those whose tiles of 256 x 256 fill every round, as its own do: 6,144 x 4,096 at
        8,192 rows 267 / 276, 4,096 x 4,096 at 4,096 88 / 93, 4,096 x 8,192 at 8,192 342 / 364, 16,384 x 2,048 at 4,096 190 / 205, 8,192 x 4,096
        at 1,800 90 / 95 (1.04 of its time over 81 sizes, a tile's front and its way out beside a walk of few steps; but 4,096 x 12,288 at 4,096
        269 / 257 and 8,192 527 / 510, and one or two rounds of at most eight steps, 8,192 x 512 at 2,048 23.8 / 21.3 and 4,096 41.5 / 40.7, 8,192
        77 / 82).  And inner dimensions of 16,384 and more in tiles of 192 x 256: 5,120 x 25,600 at 1,800 371 /
        444 and 4,096 801 / 914, 5,120 x 17,408 at 4,096 532 / 583 (in those of 256 x 256 at 2,560 562 / 311, of 192 x 192 at 1,536 351 / 214).
        Over 391 sizes of 23 weights beyond 512 rows the rule comes to 0.96 of the library's time, 27 of them by 3 to 6 % on the wrong
        side.  (The library's times jump with the rows,
        28 us at 255 and 42 at 256 for 6,144 x 4,096, so a rule of sizes leaves some on the wrong side: 5 to 15 % at a twentieth of the 375
        sizes measured up to 512 rows, 6,144 x 2,560 at 255 20 / 23, 4,608 x 3,072 at 444 25 / 29.)"""
        tile_n, tile_m = kernels.gemm_stages_tile(rows, n, k)
        tiles, units = ((n + tile_n - 1) // tile_n) * ((rows + tile_m - 1) // tile_m), compute_units()
        fill = tiles / (((tiles + units - 1) // units) * units)
        if rows <= self.STAGE_ROWS[1]:
            return fill >= 0.7 or (k <= 2048 and fill >= 0.33)
        if rows > self.STAGE_ROWS_SHARES:
            side = self.LIBRARY_TILE
            theirs = ((n + side - 1) // side) * ((rows + side - 1) // side)
            few = k <= self.STAGE_SHORT_K and theirs <= 2 * units
            if (theirs % units == 0 and k < self.STAGE_LONG_K[0] and not few) \
                    or (k >= self.STAGE_LONG_K[1] and (tile_n, tile_m) == (192, 256)):
                return False
            return kernels.gemm_stages_time(rows, n, k) * 1000 * self.STAGE_RATE <= 2 * rows * n * k
        return n <= 32 * units and (fill >= 0.95 or (fill >= 0.7 and (k <= 2048 or (k <= 4096 and tile_n * tile_m >= 96 * 128))))

    def stage_shares_for(self, x: torch.Tensor) -> int:
        """Into how many shares of the inner dimension the product in stages cuts an update that the next norm adds up; 0:
        not this product.  Up to 192 rows the cut depends on the weight's shape alone, as that of the shared-out product, so
        a row's sums do not depend on how many rows are beside it (the best cut for 128 rows: as fast as one by the rows, but
        2,560 x 4,096 at 192 rows 23 us against 19); beyond it goes with the rows."""
        rows, n, k = x.shape[0], self.out_features, self.in_features
        if not (self.library and x.dtype == torch.bfloat16 and self.STAGE_ROWS[0] <= rows and self.operands_ok(x)) \
                or n % 4 or k % 64 or (n * k < self.STAGE_MIN_WEIGHT and not self.library_shares_for(x)):
            return 0
        if rows >= self.TILE_MIN_ROWS and (OWN_MANY_ROWS == "none" or self.tile_shares_for(x)):
            return 0
        if rows > self.STAGE_ROWS_SHARES and not self.library_shares_for(x):
            return 0
        return kernels.gemm_stages_shares(self.STAGE_CUT_ROWS if rows <= self.SHARES_ROWS[1] else rows, n, k)

    PARTS_MIN_K = 4096           # a plain product's inner dimension from which on its consumer had better add shares up

    def may_part(self, rows: int) -> bool:
        """Whether a plain product of that many rows can be one in shares at all (a question for every layer of every step)."""
        return self.in_features >= self.PARTS_MIN_K and self.STAGE_ROWS[0] <= rows <= self.STAGE_ROWS_SHARES

    def parts_shares_for(self, x: torch.Tensor) -> int:
        """Into how many shares of the inner dimension a plain product is cut for a consumer that adds them up on the way (the rotation
        of q and k, ``forward_parts``); 0: it is the faster one as it is.

        The whole product has few tiles at some hundreds of rows, and a tile's walk takes as long as K is long; shares fill the chip
        and cost the consumer their way from memory.  Product and rotation, us, whole (own / the library's) / in shares: 6,144 x 4,096 at
        65 / 97 / 128 / 129 / 192 / 193 / 256 / 257 / 357 / 384 rows 23.9 / 22.0 / 25.0 / 30.0 / 29.4 / 29.3 / 32.8 / 35.7 / 37.3 / 38.6 and
        19.5 / 21.8 / 23.2 / 26.7 / 28.2 / 28.5 / 29.6 / 30.5 / 33.4 / 33.4; 7,168 x 5,120 at 65 / 129 / 256 / 387 36 / 46 / 43 / 53 and 28 / 31 /
        38 / 47; 10,240 x 8,192 at 65 / 192 / 512 78 / 67 / 101 and 49 / 54 / 89.  Of shorter inner dimensions it depends on the rows: 6,144 x 2,560
        at 65 / 97 / 160 / 357 21.4 / 19.3 / 27.4 / 30.7 and 17.0 / 19.7 / 24.9 / 32.6.

        Up to 256 rows the cut depends on the weight's shape alone, and where the whole product would be the one in stages at
        each of these rows, so does the question whether to cut: a row's sums do not depend on how many rows are beside it.  Of other
        shapes a product whose smallest tiles fill the chip once stays whole (5,120 x 4,096 at 160 rows 22.3 / 25.5).  Beyond, one whose own
        tiles fill their rounds (6,144 x 4,096 at 388 / 448 / 512 rows 38.5 / 35.6 / 39.3 and 37.1 / 36.4 / 38.5 in two shares, for
        which a row's results take twice the room), and one of so many tiles that the library's fill the chip half (18,432 x 7,168 at 300 rows
        111 / 118).  Over 425 sizes of 17 weights 0.80 of the time, five of them 3 to 7 % and one 12 % slower (most where the
        library's time jumps at 257 rows)."""
        rows, (n, k) = x.shape[0], self.weight.shape
        if not (self.may_part(rows) and self.may_stage(x, self.weight)) or n % 4:
            return 0
        tile_n, tile_m = kernels.gemm_stages_tile(rows, n, k)
        tiles, units = ((n + tile_n - 1) // tile_n) * ((rows + tile_m - 1) // tile_m), compute_units()
        if rows <= self.STAGE_ROWS[1]:
            shares = kernels.gemm_stages_shares(self.SHARES_ROWS[1], n, k)
            whole = tile_n * tile_m <= 64 * 64 and 0.9 * units <= tiles <= units and not self.always_stages(n, k, units)
        else:
            shares = kernels.gemm_stages_shares(rows, n, k)
            side = self.LIBRARY_TILE
            theirs = ((n + side - 1) // side) * ((rows + side - 1) // side)
            whole = theirs > units // 2 or (self.takes_stages(x) and tiles >= 0.9 * units * ((tiles + units - 1) // units))
        return 0 if whole or shares < 2 else shares

    def always_stages(self, n: int, k: int, units: int) -> bool:
        """Whether a plain product of this shape goes in stages at every number of rows up to 255."""
        key = (n, k, units)
        if key not in Linear._always:
            Linear._always[key] = all(self.fills_stages(rows, n, k) for rows in range(self.STAGE_ROWS[0], self.TILE_MIN_ROWS))
        return Linear._always[key]

    _always: dict = {}           # (of shapes; a function of the sizes alone)

    def forward_parts(self, x: torch.Tensor, workspace: Workspace) -> Optional[torch.Tensor]:
        """The product as float32 shares [shares, rows, out] in a buffer of the workspace, for a caller whose next kernel adds
        them up on the way, or None: it is the faster one as it is (``parts_shares_for``)."""
        shares = self.parts_shares_for(x)
        if not shares:
            return None
        rows, (n, k) = x.shape[0], self.weight.shape
        parts = workspace.buffer(f"linear.shares.{n}.{k}", shares * rows, n, torch.float32).view(shares, rows, n)
        kernels.gemm_stages(x, self.weight, parts)
        return parts

    TILE_MIN_ROWS = 256          # from here on the tiled product for many rows is a candidate, and ``OWN_MANY_ROWS`` decides

    def takes_tiles(self, x: torch.Tensor, w: Optional[torch.Tensor] = None, swiglu: bool = False) -> bool:
        """Whether a product of this many rows runs as this package's tiled product (``OWN_MANY_ROWS`` allowing)."""
        w = self.weight if w is None else w
        if OWN_MANY_ROWS in ("none", "stages") or (OWN_MANY_ROWS == "swiglu" and not swiglu):
            return False
        return (self.library and x.dtype == torch.bfloat16 and x.shape[0] >= self.TILE_MIN_ROWS and self.operands_ok(x)
                and kernels.gemm_tile_takes(x.shape[0], w.shape[0], w.shape[1], swiglu=swiglu))

    def tile_shares_for(self, x: torch.Tensor) -> int:
        """Into how many shares of the inner dimension the tiled product of many rows is cut when it adds into the
        residual (float32 results that the next norm adds up); 0: not this product.  As many shares as bring the
        tiles to the number of compute units, at most 8."""
        if OWN_MANY_ROWS != "all" or not self.takes_tiles(x) or self.out_features % 4:
            return 0
        tile = kernels.TILE_ROWS
        tiles = ((x.shape[0] + tile - 1) // tile) * ((self.out_features + tile - 1) // tile)
        splits = max(1, min(8, compute_units() // tiles))
        while splits > 1 and self.in_features % (splits * kernels.TILE_K):
            splits -= 1
        return splits

    def takes_shared_k(self, x: torch.Tensor, w: torch.Tensor, out: torch.Tensor) -> bool:
        """Whether a bfloat16 product of 17 to 64 rows runs with the inner dimension shared out inside a workgroup:
        weights of so few rows that a wavefront a slab leaves most of the chip's wavefront slots empty."""
        return (out.dtype == torch.bfloat16 and w.shape[0] <= 32 * compute_units()
                and kernels.gemm_rows_takes(x.shape[0], w.shape[0], w.shape[1]))

    def takes_mid(self, x: torch.Tensor) -> bool:
        return (self.library and x.dtype == torch.bfloat16 and self.MID_ROWS[0] <= x.shape[0] <= self.MID_ROWS[1]
                and self.operands_ok(x) and self.swiglu_waves_for(x.shape[0]) > 0)

    def swiglu_waves_for(self, rows: int) -> int:
        """Wavefronts a workgroup of the product for 17 to 64 rows with SwiGLU inside (no sharing out of the inner
        dimension there), or 0 where the library's product followed by the SwiGLU kernel is faster.

        The estimate is again the fullest compute unit's: workgroups on it x (weight rows a workgroup + half the
        rows of X, which every workgroup fetches).  Measured at 32 rows: 8B shape (24,576 weight rows) 96 rows a
        workgroup 37.9 us (one workgroup a unit), 64 rows 43.6; 14B shape (34,816) 160 rows 68.8 us, 96 rows 80.5
        (363 workgroups: two on some units); 32B shape (51,200) 64 rows 117 us, the best of all shapes, against
        the library's 100 + 5: no shape shares 200 rows a unit out evenly, so the library takes that one (the rule:
        this product's estimate must stay below 1.5 x the weight rows a unit)."""
        n = self.out_features
        units = compute_units()
        if n <= 32 * units:
            return 2    # too few weight rows to fill the chip in any shape: the most workgroups
        best = None
        for waves in (2, 4, 6, 10):
            on_a_unit = ((n + 16 * waves - 1) // (16 * waves) + units - 1) // units
            cost = on_a_unit * (16 * waves + rows // 2)
            if best is None or cost < best[0]:
                best = (cost, waves)
        if n <= 64 * units:
            return best[1]    # (12,288 weight rows: 64 rows a workgroup 12 to 15 us, the library 15 to 18 + 5)
        return best[1] if best[0] * units < 1.5 * n else 0

    def shares_for(self, x: torch.Tensor) -> int:
        """Into how many shares the inner dimension is cut for an update in parts; 0: not this product."""
        return self.shares_and_waves_for(x)[0]

    def shares_and_waves_for(self, x: torch.Tensor):
        """(shares of the inner dimension, wavefronts a workgroup) of the product for 17 to 192 rows whose float32
        partial results the next norm adds up; (0, 0): not this product.

        The pair with the least estimated time of the fullest compute unit is taken: workgroups on it (all of them
        over the compute units, rounded up) x weight rows a workgroup x (length of a share + 280, what a workgroup costs
        beside its walk), plus half a microsecond a share for the norm that adds them up.  Measured at 64 rows: down
        of the 8B shape 4 shares of 64 rows (256 workgroups) 23.8 us, 8 shares 24.9, 6 shares (384 workgroups, two on
        half the units) 28.6; down of the 14B shape 4 shares of 96 rows (216 workgroups) 40.9 us, 8 shares of 64 rows
        (640 workgroups) 46.9."""
        if not (self.library and x.dtype == torch.bfloat16 and self.SHARES_ROWS[0] <= x.shape[0] <= self.SHARES_ROWS[1]
                and self.operands_ok(x)) or self.out_features % 4:
            return 0, 0
        best = None
        units = compute_units()
        for waves in (4, 6):
            rows = 16 * waves
            tiles = (self.out_features + rows - 1) // rows
            for splits in range(1, 17):
                if self.in_features % splits or (self.in_features // splits) % 128:
                    continue
                share = self.in_features // splits
                on_a_unit = (tiles * splits + units - 1) // units
                cost = on_a_unit * rows * (share + 280) + 8000 * splits
                if best is None or cost < best[0]:
                    best = (cost, splits, waves)
        return (best[1], best[2]) if best else (0, 0)

