"""y = x . W^T (+ b): the matrix product every part uses."""

from __future__ import annotations

from typing import Optional

import torch

from .. import ops
from ..ops.tuning import library_mm, library_tuning_enabled
from ..ops.functions import (GEMM_MFMA_SKINNY_BEST_M, GEMM_MFMA_SKINNY_MAX_M, GEMM_MFMA_WIDE_MAX_M,
                             GEMM_SKINNY_MAX_M)


class Linear:
    """Holds ``weight`` [N, K] in the compute dtype and an optional float32 ``bias`` [N].

    float32: the engine's own kernels only (true 32-bit products and sums): vector FMA kernels for 1 and 2
    rows, and from 3 rows on the matrix cores' float32 instruction, which rounds nothing: a kernel that
    streams W up to 64 rows, one of 64 x 64 tiles beyond; residual projections leave partial sums.  A weight of 2 MB and more
    has a second copy in the order of that instruction's fragments (``streamed32``), from which a third kernel takes up to
    64 rows, one and two among them (``ops.gemm_fp32_stream_plan``).
    bfloat16: up to 16 rows (decoding) the engine's matrix-core kernel that streams the weight
    once; its sibling that shares x through LDS for float32 results of 8 to 64 rows (the logits;
    beyond 64 rows the library with a float32 result), for the residual projections
    (``for_residual``: 17 to 64 rows, and any number where K is long) and for the partial sums of
    other projections of 17 to 64 rows (``partial_sums``); a third for up to 16 rows and a K so short that all of it is under
    way at once (``ops.gemm_stream_plan``); residual projections of more than 128 rows whose K is 16,384
    and more the engine's kernel for many rows, in slices of K (``ops.gemm_tile_plan``); products of 17 rows
    and more that no other of these takes, of matrices up to some 50 MB, the one in small tiles (``ops.gemm_block_plan``, up to 64 rows
    those of a short K or few rows of W: ``partial_sums``); everything else
    the library product (hipBLASLt through torch, where the reference's engine calls cuBLAS) with
    float32 accumulation, the bias added by a kernel of the engine.  A large weight has a second copy in
    the order of the matrix instruction's fragments (``prepare``, ``streamed``), from which the
    sibling takes every product of up to 64 rows.

    The copies hold what the weight was when ``prepare`` ran: setting ``weight`` drops them, and after a change of the weight's
    values in place ``prepare`` is called again (or ``drop_copy``), in either precision."""

    narrow_to = 64  # float32 results of at most this many outputs from bfloat16 operands: the narrow kernel
    float32_on_matrix_cores = True  # 3 rows of float32 and more: v_mfma_f32_16x16x4_f32 instead of vector FMAs
    # A bfloat16 weight of at least this many bytes is kept a second time, in the order of the matrix
    # instruction's fragments, for the engine's own products (decoding): a wave then loads 1 KB in one
    # piece with streaming loads, where rows give it 16 pieces of 64 bytes (a compute unit draws about
    # half as much when a wave's load is pieces of rows).  From 8 MB on (8 rows: N = 896, K = 4864, 8.7 MB,
    # 4.2 us against 4.8; N = K = 2048 3.7 / 4.2; N = 3072, K = 2048 4.2 / 4.9; below that a launch is most of
    # the time).  The rows stay for the library's products of many rows.  None: no copies.
    # A copy that would leave less than ``streamed_copy_reserve`` of the device's memory free is not
    # made: a model that large keeps copies of its first layers only and runs the rest from rows.
    # Up to 64 rows read any copy: 0.86 to 1.0 of the time from rows at 15 sizes of 8 to 15 MB, with the norm.  (A model of few layers
    # has such matrices in the Infinity Cache as rows, which the copies' streaming loads pass by: steps of 20 rows of
    # 8 layers at hidden size 2,048 13.2 ms of 24 from copies, 13.1 from rows, but of 28 layers 41.8 and 43.3, 32 layers at 2,560 50.4 and
    # 51.6; the 0.5B shape, 64 rows, 29.3 and 30.7.)  Beyond 64 rows copies of 16 MB and more are read: those of 8 to 16 MB are no
    # faster than the library's product there.  (Where ``streamed_copy_from`` is set lower, from twice that size on.)
    streamed_copy_from = 8 << 20
    streamed_many_rows_from = 16 << 20
    streamed_copy_reserve = 0.25
    # A float32 weight from this size on (where copies are made at all): 4 rows of N = K = 896, 3.2 MB, 2.7 us against 3.5; N = 1152 3.1 / 4.1
    streamed32_copy_from = 2 << 20

    def __init__(self, in_features: int, out_features: int, bias: bool = False):
        self.in_features = in_features
        self.out_features = out_features
        self.has_bias = bias
        self._weight: Optional[torch.Tensor] = None
        self.bias: Optional[torch.Tensor] = None
        self.streamed = None  # the weight in fragment order (ops.FragmentOrdered), if prepare() made one
        self.streamed32 = None  # the same of a float32 weight
        self._wide_splits: dict = {}  # tiles of rows -> slices of K (a property of the sizes alone)
        self._wide_takes: dict = {}   # (tiles, slices, gate/up) -> whether the kernel takes them from this weight
        self._many_plans: dict = {}   # (rows, result, library tuning) -> how a product of more than 16 rows is taken (of the sizes alone)

    @property
    def weight(self) -> Optional[torch.Tensor]:
        return self._weight

    @weight.setter
    def weight(self, t: Optional[torch.Tensor]) -> None:
        self._weight = t
        self.streamed32 = None
        self.streamed = None  # a copy of the weight that was here says nothing about this one
        self._wide_takes = {}

    def prepare(self, copies: bool = True) -> None:
        """Called by the owning part once the weight is set.  ``copies=False``: no second copy."""
        w = self.weight
        self.streamed = self.streamed32 = None
        if not copies or self.streamed_copy_from is None or w is None or not w.is_cuda:
            return
        size = w.numel() * w.element_size()
        if w.dtype == torch.bfloat16:
            wanted = size >= self.streamed_copy_from and ops.gemm_mfma_wide_splits_ok(self.in_features, 1)
        else:
            wanted = (w.dtype == torch.float32 and size >= self.streamed32_copy_from and w.is_contiguous() and w.data_ptr() % 16 == 0
                      and ops.gemm_fp32_stream_plan(4, self.out_features, self.in_features, ops.GEMM_FP32_SUMS) is not None)
        if not wanted:
            return
        free, total = torch.cuda.mem_get_info(w.device)
        if free - size >= self.streamed_copy_reserve * total:
            if w.dtype == torch.bfloat16:
                self.streamed = ops.fragment_order(w)
            else:
                self.streamed32 = ops.fragment_order(w)

    def kernel_reads(self, x: torch.Tensor) -> bool:
        """Whether the engine's 16-byte loads can read ``x`` and the weight as they lie: rows without gaps, on 16 bytes.
        Where not, a product of many rows goes to the library or the vector kernels, which take any."""
        w = self._weight
        return x.is_contiguous() and x.data_ptr() % 16 == 0 and w.is_contiguous() and w.data_ptr() % 16 == 0

    def takes_f32_matrix(self, x: torch.Tensor) -> bool:
        """Whether a whole float32 product of these rows runs on the matrix cores."""
        return (self.float32_on_matrix_cores and x.shape[0] > 2 and self.in_features % 4 == 0
                and (x.shape[0] <= GEMM_MFMA_SKINNY_MAX_M or self.kernel_reads(x)))

    def drop_copy(self) -> int:
        """Forget the fragment-ordered copy (the products then read rows); returns its bytes."""
        freed = sum(c.data.numel() * c.data.element_size() for c in (self.streamed, self.streamed32) if c is not None)
        self.streamed = self.streamed32 = None
        self._wide_takes = {}
        return freed

    def sums32(self, x: torch.Tensor) -> Optional[torch.Tensor]:
        """x . W^T (no bias) of float32 rows as partial sums [S, T, N] (S = 1 where the product is better left whole) from the copy, or None."""
        plan = self.plan32(x, ops.GEMM_FP32_SUMS)
        if plan is None:
            return None
        y = ops.gemm_fp32_stream(x, self.streamed32, plan)
        return y if y.ndim == 3 else y.unsqueeze(0)

    def plan32(self, x: torch.Tensor, result: int) -> Optional[int]:
        """How the float32 kernel of the fragment-ordered copy takes ``x`` (``ops.gemm_fp32_stream``), or None."""
        m = x.shape[0]
        if self.streamed32 is None or not 0 < m <= GEMM_MFMA_SKINNY_MAX_M or not self.float32_on_matrix_cores or not self.kernel_reads(x):
            return None
        return ops.gemm_fp32_stream_plan(m, self.out_features, self.in_features, result)

    def copy_for(self, m: int):
        """The fragment-ordered copy, if there is one that products of ``m`` rows read."""
        if self.streamed is None or m <= GEMM_MFMA_SKINNY_MAX_M:
            return self.streamed
        least = min(self.streamed_many_rows_from, 2 * (self.streamed_copy_from or 0))
        return self.streamed if self._weight.numel() * 2 >= least else None

    def wide_weight(self, m: int):
        """What the products of ``m`` rows that share x through LDS read: the fragment-ordered copy if there is one for them."""
        copy = self.copy_for(m)
        return self.weight if copy is None else copy

    def __call__(self, x: torch.Tensor, out_dtype: Optional[torch.dtype] = None,
                 skip_bias: bool = False) -> torch.Tensor:
        bias = None if skip_bias else self.bias
        w = self.weight
        m = x.shape[0]
        if m > GEMM_MFMA_WIDE_MAX_M and out_dtype is None and x.dtype == torch.bfloat16 and not (self.in_features % 8 or self.out_features % 8):
            return self._many_rows(x, bias)
        if x.dtype == torch.float32:
            plan = self.plan32(x, ops.GEMM_FP32_WHOLE) if out_dtype in (None, x.dtype) else None
            if plan is not None:
                return ops.gemm_fp32_stream(x, self.streamed32, plan, bias)
            if self.float32_on_matrix_cores and 2 < m <= GEMM_MFMA_SKINNY_MAX_M and self.in_features % 4 == 0:
                # decoding in the 32-bit path: W streams once into true float32 matrix instructions
                # (several times faster than the vector kernels from 8 rows on, no faster at one or two)
                return ops.gemm_mfma_fp32(x, w, bias)
            if (self.float32_on_matrix_cores and m > GEMM_MFMA_SKINNY_MAX_M and self.in_features % 4 == 0
                    and self.kernel_reads(x) and out_dtype in (None, x.dtype)):
                return ops.gemm_fp32_tile(x, w, bias)  # prompts: the same instruction, both operands through LDS
            return ops.gemm(x, w, bias, out_dtype=out_dtype)
        wants_f32 = out_dtype is not None and out_dtype != x.dtype
        if wants_f32 and out_dtype == torch.float32 and self.out_features <= self.narrow_to:
            # a handful of float32 outputs a row (gates): a wave a row, the matrix from cache
            return ops.gemm(x, w, bias, out_dtype=out_dtype, kind=ops.GEMM_NARROW)
        if (wants_f32 and bias is None and (8 if self.streamed is None else 1) <= m <= GEMM_MFMA_SKINNY_MAX_M
                and ops.gemm_mfma_wide_splits_ok(self.in_features, 1)):
            # float32 results (logits) of 8 to 64 rows: x shared through LDS; from the fragment-ordered
            # copy at any number of rows
            return ops.gemm_mfma_wide(x, self.wide_weight(m))
        if (wants_f32 and bias is None and m > GEMM_MFMA_SKINNY_MAX_M and out_dtype == torch.float32
                and self.in_features % 8 == 0 and self.out_features % 8 == 0):
            # logits of more rows than the engine's kernels take (a decode batch beyond 64, a replay
            # that wants every position): the library with a float32 result
            return library_mm(x, w, float32_result=True)
        if not wants_f32 and 0 < m <= GEMM_MFMA_SKINNY_BEST_M:
            plan = self.stream_plan(m, ops.GEMM_STREAM_POINT)
            if plan is not None and self.kernel_reads(x):
                return ops.gemm_mfma_stream(x, self.wide_weight(m), ops.GEMM_STREAM_POINT, plan, bias)
        if self.in_features % 8 == 0 and m <= (GEMM_MFMA_SKINNY_MAX_M if wants_f32 else GEMM_MFMA_SKINNY_BEST_M):
            return ops.gemm_mfma_skinny(x, w, bias, out_dtype=out_dtype)
        if not wants_f32 and self.out_features % 4 == 0:
            # 17 to 64 rows (to 128 from a fragment-ordered copy): the engine's product that shares x through LDS, as
            # float32 partial sums of slices of K, added up and rounded once; the library needs 40 us for 64 rows of
            # a matrix whose read is 8 us
            sums = self.partial_sums(x)
            if sums is not None:
                return ops.sum_round(sums, bias)
        if m <= GEMM_SKINNY_MAX_M or wants_f32 or self.in_features % 8 or self.out_features % 8:
            # few rows with an odd inner size; float32 results from bfloat16 operands (logits of
            # many rows); and sizes whose rows are not 16-byte aligned, which the library is not given
            return ops.gemm(x, w, bias, out_dtype=out_dtype)
        return self._many_rows(x, bias)

    def _many_plan(self, m: int, result: int):
        """(tile, slices of K, whether it is the kernel for many rows; else the small tiles') for ``m`` rows, or None where the library's
        product is the better one.  Remembered by the rows: a property of the sizes alone, asked for in every layer and step."""
        # (the library's kernels chosen by timing: every product that is not the large kernel's is then the library's, which a program asks for
        # that way, though the small tiles took 0.50 to 0.88 of the timed kernels' time at 17 of 19 sizes, 1.02 at two)
        tuned = library_tuning_enabled()
        key = (m, result, tuned)
        if key not in self._many_plans:
            if len(self._many_plans) > 1024:
                self._many_plans.clear()
            n, k = self.out_features, self.in_features
            large = ops.gemm_tile_plan(m, n, k, ops.GEMM_TILE_SUMS) if result == ops.GEMM_BLOCK_SUMS and m > GEMM_MFMA_WIDE_MAX_M else None
            if large is not None:
                plan = None if large[1] == 1 and tuned else large + (True,)
            else:
                plan = None if tuned else ops.gemm_block_plan(m, n, k, result)
                # (a whole product is better left in bfloat16, half the bytes for the norm)
                plan = None if plan is None or (result == ops.GEMM_BLOCK_SUMS and plan[1] == 1) else plan + (False,)
            self._many_plans[key] = plan
        return self._many_plans[key]

    def _many_rows(self, x: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
        plan = self._many_plan(x.shape[0], ops.GEMM_BLOCK_PLAIN)
        if plan is not None and self.kernel_reads(x) and (bias is None or bias.data_ptr() % 16 == 0):
            return ops.gemm_mfma_block(x, self._weight, ops.GEMM_BLOCK_PLAIN, plan[0], bias=bias)
        y = library_mm(x, self._weight)
        if bias is not None:
            ops.bias_add(y, bias)
        return y

    def for_residual(self, x: torch.Tensor, ctx) -> torch.Tensor:
        """The product as the delta of the residual stream.  For a few rows (decoding) and a
        long inner dimension the matrix-core kernel cuts K into slices with workgroups of their
        own, which fills the chip where N alone leaves too few of them, and returns their float32
        partial sums [S, T, N]; the next norm adds them up in order."""
        sums = self.residual_sums(x, ctx)
        return self(x) if sums is None else sums

    def for_stream(self, x: torch.Tensor, ctx) -> torch.Tensor:
        """The same for a delta that is the whole stream: never rounded to 16 bits (partial sums, or [T, N] in float32)."""
        sums = self.residual_sums(x, ctx)
        return self(x, out_dtype=torch.float32) if sums is None else sums

    def residual_sums(self, x: torch.Tensor, ctx) -> Optional[torch.Tensor]:
        """The partial sums of ``for_residual``, or None where the product is better left whole."""
        if self.bias is not None or not getattr(ctx, "partial_sums_ok", False):
            return None
        m = x.shape[0]
        if x.dtype == torch.float32:
            # the 32-bit path: slices of K where the rows of W alone (or a prompt's tiles) leave the chip idle
            sums = self.sums32(x)
            if sums is not None:
                return sums
            if not self.float32_on_matrix_cores or m <= 2 or self.in_features % 4:
                return None
            if m <= GEMM_MFMA_SKINNY_MAX_M:
                splits = ops.gemm_mfma_fp32_splits(self.in_features, self.out_features)
                return ops.gemm_mfma_fp32_sums(x, self.weight, splits) if splits > 1 else None
            splits = ops.gemm_fp32_tile_splits(m, self.out_features, self.in_features)
            return ops.gemm_fp32_tile(x, self.weight, splits=splits) if splits > 1 and self.kernel_reads(x) else None
        if x.dtype != torch.bfloat16 or m == 0:
            return None
        if m > GEMM_MFMA_WIDE_MAX_M:
            return self._many_sums(x)
        if m > GEMM_MFMA_SKINNY_MAX_M:
            # 65 to 128 rows of a fragment-ordered weight: the same kernel with five to eight tiles of x,
            # where its launch shape has one
            splits = self.wide_splits(m) if self.copy_for(m) is not None else 1
            if splits > 1 and self.wide_takes(m, splits):
                return ops.gemm_mfma_wide(x, self.streamed, splits=splits) if self.kernel_reads(x) else None
            return self._many_sums(x)
        if self.in_features % 8:
            return None
        if getattr(ctx, "sums_in_one", False):
            plan = ops.gemm_stream_plan(m, self.out_features, self.in_features, ops.GEMM_STREAM_PLAN_ONE, self.streamed is not None)
            if plan is not None and self.kernel_reads(x):
                return ops.gemm_mfma_stream(x, self.weight, ops.GEMM_STREAM_SUMS, plan)
        plan = self.stream_plan(m, ops.GEMM_STREAM_SUMS) if m <= GEMM_MFMA_SKINNY_BEST_M else None
        if plan is not None and self.kernel_reads(x):
            return ops.gemm_mfma_stream(x, self.streamed, ops.GEMM_STREAM_SUMS, plan)
        # the kernel that shares x through LDS: above 16 rows, and at any number of rows where
        # K is long enough for six slices or more
        splits = self.wide_splits(m)
        if splits > 1 and (self.kernel_reads(x) if m > GEMM_MFMA_SKINNY_BEST_M
                           else self.streamed is not None or self.slices_beat_few_rows(splits)):
            return ops.gemm_mfma_wide(x, self.wide_weight(m), splits=splits)
        splits = self.residual_splits(m)
        return ops.gemm_mfma_skinny(x, self.weight, splits=splits) if splits > 1 else None

    def _many_sums(self, x: torch.Tensor) -> Optional[torch.Tensor]:
        """Partial sums of more than 64 rows, where slices of K are faster than a whole product: a long K in the kernel for many rows (whole,
        it is no faster than the library's timed kernels: 4,096 rows of N = 3584, K = 18944 with the norm 443 us, 401; the library's own
        choice 567), else in the small tiles' one."""
        plan = self._many_plan(x.shape[0], ops.GEMM_BLOCK_SUMS)
        if plan is None or not self.kernel_reads(x):
            return None
        if plan[2]:
            return ops.gemm_mfma_tile(x, self._weight, splits=plan[1], tile=plan[0])
        return ops.gemm_mfma_block(x, self._weight, ops.GEMM_BLOCK_SUMS, plan[0], plan[1])

    def partial_sums(self, x: torch.Tensor, few_rows: bool = False, long_slices: bool = False) -> Optional[torch.Tensor]:
        """x . W^T (no bias) of 17 to 64 rows (to 128 from a fragment-ordered copy) as float32 partial
        sums [S, T, N] of slices of K, for a consumer that adds them up itself; None where the engine's
        kernel for that does not take the sizes.  ``few_rows``: also for up to 16 rows.  ``long_slices``: only in
        slices of 512 values of K and more, for a consumer to whom a slice more costs what shorter ones bring."""
        m = x.shape[0]
        most = GEMM_MFMA_SKINNY_MAX_M if self.copy_for(m) is None else GEMM_MFMA_WIDE_MAX_M
        least = 0 if few_rows else GEMM_MFMA_SKINNY_BEST_M  # (fewer rows: for a consumer that spares a launch by it)
        if x.dtype != torch.bfloat16 or not least < m <= most:
            return None
        if m > GEMM_MFMA_SKINNY_BEST_M and self.in_features < 2 * 512 and (self.in_features < 7 * 128 or self.out_features < 1024):
            # slices of one stage of K: added up by a launch of their own they pay from seven slices and 1,024 rows of W on
            # (N = 1024, K = 896: 17 rows 6.2 us, 64 8.0, the library's 6.6 and 10.4; K = 768: 5.8 and 7.3 against 5.0 and 7.0)
            return None
        splits = self.long_splits() if long_slices and m <= GEMM_MFMA_SKINNY_BEST_M else self.wide_splits(m)
        if splits < 2 or (long_slices and self.in_features < 2 * 512) or not self.wide_takes(m, splits):
            return None
        if m > GEMM_MFMA_SKINNY_BEST_M and not self.kernel_reads(x):
            return None  # (the library's)
        return ops.gemm_mfma_wide(x, self.wide_weight(m), splits=splits)

    def stream_plan(self, m: int, result: int):
        """How the kernel for few rows and a short K takes ``m`` rows of this weight, or None."""
        return ops.gemm_stream_plan(m, self.out_features, self.in_features, result, self.streamed is not None)

    def wide_takes(self, m: int, splits: int, gate_up: bool = False) -> bool:
        """Whether the kernel that shares x through LDS takes ``m`` rows of this weight (beyond 64 rows
        it has kernels for some launch shapes only)."""
        weight = self.wide_weight(m)
        key = (-(-m // 16), splits, gate_up, weight is self.streamed)
        if key not in self._wide_takes:
            self._wide_takes[key] = ops.gemm_mfma_wide_takes(m, weight, splits, gate_up)
        return self._wide_takes[key]

    def wide_splits(self, m: int) -> int:
        """Slices of K for the kernel that shares x through LDS, by the tiles of 16 rows that ``m``
        rows make (the kernel's own rule: as many as K gives, up to 8, for up to 16 rows; from 17
        rows on the cut that gives the most workgroups the device has room for).  1 = it does
        not take this K."""
        tiles = -(-m // 16)
        if tiles not in self._wide_splits:
            self._wide_splits[tiles] = ops.gemm_mfma_wide_best_splits(m, self.out_features, self.in_features)
        return self._wide_splits[tiles]

    def long_splits(self) -> int:
        """Up to eight slices of 512 values of K and more (1: K gives none)."""
        return next((s for s in range(8, 1, -1) if self.in_features >= 512 * s and ops.gemm_mfma_wide_splits_ok(self.in_features, s)), 1)

    def slices_beat_few_rows(self, splits: int) -> bool:
        """Up to 16 rows of a weight without a copy: whether the kernel that shares x through LDS, in ``splits`` slices of K,
        is faster than the few-rows kernel in two, four or eight.  Six slices or more, of 512 and more values of K; or shorter
        ones that the other kernel has no even cut for, as long as the workgroups are not too many (with the norm, 8 rows, us,
        this kernel / the other: N = K = 896 5.6 / 6.4, N = 3072, K = 896 7.6 / 7.8, N = 3584 8.1 / 8.0; N = K = 1536
        7.5 / 8.1).  At K = 1024 the other's halves are as good from N = 1,536 on (16 rows 7.4 / 7.0, N = 1024 6.0 / 6.4), and
        at K = 2048 its quarters at any N (N = 512 6.2 / 6.1, N = 1024 6.7 / 6.5)."""
        if splits < 6:
            return False
        groups = -(-self.out_features // 64) * splits
        if self.in_features < 2048:
            return groups <= (128 if self.in_features == 1024 else 384)
        return self.in_features >= 6 * 512

    def residual_splits(self, m: int) -> int:
        """Slices of K for ``for_residual`` (1 = do not cut): as many as bring the workgroups to
        about three and a half per compute unit, each slice at least 512 long.  Above 16 rows only
        where K gives four slices of 1024; shorter products of that many rows are the library's."""
        groups = -(-self.out_features // 16)
        shortest = 512 if m <= GEMM_MFMA_SKINNY_BEST_M else 1024
        splits = 1
        # (about three and a half workgroups a compute unit)
        while splits < 8 and 2 * groups * splits < 7 * ops.compute_units() and self.in_features // (2 * splits) >= shortest:
            splits *= 2
        if m > GEMM_MFMA_SKINNY_BEST_M and splits < 4:
            return 1
        return splits
