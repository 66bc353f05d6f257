"""Kernel registry over the gfx950 kernel table.

Same selection contract as the reference's KernelRegistry (registry.py:254-352):
candidates must match dtype, scale spec, epilogue, layout and schedule, be
even-K, obey the split rule, and (for ``select``) accept the shape as a tile
multiple; among them the one with the largest (measured_tops or 0,
BLOCK_M * BLOCK_N) wins, the first on ties.  measured_tops is the table's
figure for the request's shape (kernel_table.selection_tops) unless a caller
set another.  The entries come from the gfx950
kernel table (``kernel_table.TABLE``) instead of gfx1151 tile seeds: every
dense table entry is registered once per epilogue and subchannel size it
serves.
"""

from __future__ import annotations

from dataclasses import replace
from typing import Iterable

from . import kernel_table as kt
from .metadata import (
    ACC_DTYPE,
    ARCH,
    SCALE_DTYPE_BF16,
    SUPPORTED_SUBCHANNELS,
    Epilogue,
    GemmLayout,
    KernelMetadata,
    KernelSchedule,
    KernelStatus,
    OperandDType,
    ScaleMode,
    ScaleSpec,
    TileConfig,
    make_kernel_id,
    output_dtype_for_split_k,
)
from .template_config import slices_k

_LAYOUT_OF_CODE = {kt.LAYOUT_NN: GemmLayout.NN, kt.LAYOUT_NT: GemmLayout.NT, kt.LAYOUT_TN: GemmLayout.TN,
                   kt.LAYOUT_TT: GemmLayout.TT}


def _tile_of(desc: kt.KernelDesc) -> TileConfig:
    return TileConfig(
        block_m=desc.block_m,
        block_n=desc.block_n,
        block_k=desc.block_k,
        group_size_m=desc.group_size_m,
        num_warps=desc.num_waves,
        num_stages=desc.num_stages,
        waves_per_eu=max(1, desc.num_waves // 4),
        even_k=True,
        split_k=desc.split_k,
    )


def _scales_of(desc: kt.KernelDesc) -> tuple[ScaleSpec, ...]:
    if desc.scale_mode == kt.SCALE_PER_CHANNEL:
        return (ScaleSpec(ScaleMode.PER_CHANNEL),)
    return tuple(
        ScaleSpec(ScaleMode.SUBCHANNEL, s)
        for s in SUPPORTED_SUBCHANNELS
        if desc.min_subchannel <= s <= desc.max_subchannel
    )


def _epilogues_of(desc: kt.KernelDesc) -> tuple[Epilogue, ...]:
    if desc.epilogue_kind == kt.EPI_KIND_SWIGLU:
        return (Epilogue.SWIGLU,)
    if desc.schedule == kt.SCHEDULE_PERSISTENT or desc.split_k > 1:
        return (Epilogue.NONE,)  # the reference's persistent kernels (registry.py:230-251)
    return (Epilogue.NONE, Epilogue.RELU2)


def iter_supported_kernel_metadata() -> Iterable[KernelMetadata]:
    """One KernelMetadata per (dense table entry, epilogue, scale spec)."""
    for desc in kt.entries(kt.FAMILY_DENSE):
        dtype = OperandDType.INT4 if desc.dtype_bits == 4 else OperandDType.INT8
        tile = _tile_of(desc)
        layout = _LAYOUT_OF_CODE[desc.layout]
        for scale in _scales_of(desc):
            for epilogue in _epilogues_of(desc):
                schedule = (KernelSchedule.PERSISTENT if desc.schedule == kt.SCHEDULE_PERSISTENT
                            else KernelSchedule.STANDARD)
                kernel_id = make_kernel_id(dtype, scale, epilogue, tile, arch=ARCH, layout=layout, schedule=schedule)
                yield KernelMetadata(
                    kernel_id=kernel_id,
                    arch=ARCH,
                    a_dtype=dtype,
                    b_dtype=dtype,
                    acc_dtype=ACC_DTYPE,
                    output_dtype=output_dtype_for_split_k(tile.split_k),
                    scale_dtype=SCALE_DTYPE_BF16,
                    scale=scale,
                    epilogue=epilogue,
                    tile=tile,
                    triton_kernel_name=f"shk::dense_gemm_kernel#{desc.index}",
                    layout=layout,
                    schedule=schedule,
                    assembly_path=None,
                    status=KernelStatus.COMPILED,
                    table_index=desc.index,
                    measured_tops=kt.measured_tops(desc),
                )


class _Candidate:
    """A kernel of a family with what decides whether it runs a shape: the
    multiples of the launch-shape contract (template_config.py
    tile_multiple_rejection_reasons) and its K bound, as plain numbers."""

    __slots__ = ("kernel", "desc", "split_k", "block_m", "block_n", "period", "sub", "slice_sub", "max_k", "table_figure",
                 "area")

    def __init__(self, kernel: KernelMetadata) -> None:
        tile = kernel.tile
        self.kernel = kernel
        self.desc = None if kernel.table_index is None else kt.TABLE[kernel.table_index]
        self.split_k = tile.split_k
        self.block_m, self.block_n, self.period = tile.block_m, tile.block_n, tile.block_k * tile.split_k
        subchannel = kernel.scale.mode is ScaleMode.SUBCHANNEL and kernel.scale.subchannel_size is not None
        self.sub = kernel.scale.subchannel_size if subchannel else 1
        self.slice_sub = self.sub if subchannel and tile.split_k > 1 and slices_k(kernel) else 1
        # the library's bound (gfx950 accumulators and buffer offsets)
        self.max_k = None if self.desc is None else self.desc.max_k
        # whether measured_tops is the table's, not a caller's own (with_status)
        self.table_figure = self.desc is not None and kernel.measured_tops == kt.measured_tops(self.desc)
        self.area = None if self.desc is not None and self.desc.plans_rows else tile.block_m * tile.block_n

    def accepts(self, m: int, n: int, k: int) -> bool:
        return not (m % self.block_m or n % self.block_n or k % self.period or k % self.sub
                    or k // self.split_k % self.slice_sub) and (self.max_k is None or k <= self.max_k)


def _selection_key(c: _Candidate, m: int, n: int | None = None, k: int | None = None) -> tuple[float, int]:
    tops = c.kernel.measured_tops
    if c.table_figure:
        tops = kt.selection_tops(c.desc, m, n, k, c.kernel.scale.subchannel_size)
    return (tops or 0.0, c.area or kt.selection_area(c.desc, m))


class KernelRegistry:
    def __init__(self, kernels: Iterable[KernelMetadata] = ()) -> None:
        self._kernels: dict[str, KernelMetadata] = {}
        # Selections are memoized per request (mm() selects on every call, and
        # a scan of the table costs hundreds of microseconds); the candidates
        # are indexed by family.  register() clears both.
        self._families: dict[tuple, list[KernelMetadata]] | None = None
        self._selected: dict[tuple, KernelMetadata] = {}
        self._call_kernels: dict[tuple, KernelMetadata] = {}
        for kernel in kernels:
            self.register(kernel)

    def register(self, kernel: KernelMetadata) -> None:
        if kernel.kernel_id in self._kernels:
            raise ValueError(f"duplicate kernel id: {kernel.kernel_id}")
        self._kernels[kernel.kernel_id] = kernel
        self._families = None
        self._selected = {}
        self._call_kernels = {}

    def _family(self, dtype, scale, epilogue, layout, schedule) -> list[_Candidate]:
        families = self._families
        if families is None:
            families = {}
            for kern in self._kernels.values():
                if kern.a_dtype is not kern.b_dtype or not kern.tile.even_k:
                    continue
                if kern.epilogue in {Epilogue.RELU2, Epilogue.SWIGLU} and kern.tile.split_k != 1:
                    continue
                key = (kern.a_dtype, kern.scale, kern.epilogue, kern.layout, kern.schedule)
                families.setdefault(key, []).append(_Candidate(kern))
            self._families = families
        return families.get((dtype, scale, epilogue, layout, schedule), [])

    def get(self, kernel_id: str) -> KernelMetadata:
        return self._kernels[kernel_id]

    def all(self) -> tuple[KernelMetadata, ...]:
        return tuple(self._kernels.values())

    def select(
        self,
        *,
        dtype: OperandDType,
        scale: ScaleSpec,
        epilogue: Epilogue,
        m: int,
        n: int,
        k: int,
        layout: GemmLayout = GemmLayout.NN,
        split_k: int | None = None,
        schedule: KernelSchedule = KernelSchedule.STANDARD,
        require_compiled: bool = False,
    ) -> KernelMetadata:
        request = (dtype, scale, epilogue, m, n, k, layout, split_k, schedule, require_compiled)
        hit = self._selected.get(request)
        if hit is not None:
            return hit
        candidates = [
            c for c in self._family(dtype, scale, epilogue, layout, schedule)
            if (split_k is None or c.split_k == split_k) and c.accepts(m, n, k)
        ] if m > 0 and n > 0 and k > 0 else []
        if require_compiled:
            candidates = [c for c in candidates
                          if c.kernel.status in {KernelStatus.COMPILED, KernelStatus.BENCHMARKED}]
        if not candidates:
            raise LookupError(
                f"no kernel for dtype={dtype.value}, scale={scale.label}, epilogue={epilogue.value}, "
                f"layout={layout.value}, schedule={schedule.value}, shape=({m}, {n}, {k})"
            )
        chosen = max(candidates, key=lambda c: _selection_key(c, m, n, k)).kernel
        if len(self._selected) >= 4096:  # bounded for callers that vary M call to call
            self._selected = {}
        self._selected[request] = chosen
        return chosen

    def select_call(
        self,
        *,
        dtype: OperandDType,
        scale: ScaleSpec,
        epilogue: Epilogue,
        m: int,
        n: int,
        k: int,
        layout: GemmLayout = GemmLayout.NN,
        split_k: int | None = None,
        schedule: KernelSchedule = KernelSchedule.STANDARD,
    ) -> KernelMetadata:
        """The kernel that a whole call of a request runs: call_kernel of what
        select() picks, in one memo lookup a call."""
        request = (dtype, scale, epilogue, m, n, k, layout, split_k, schedule)
        hit = self._call_kernels.get(request)
        if hit is not None:
            return hit
        chosen = self.call_kernel(
            self.select(dtype=dtype, scale=scale, epilogue=epilogue, m=m, n=n, k=k, layout=layout, split_k=split_k,
                        schedule=schedule), m=m, n=n, k=k)
        if getattr(self.select, "__func__", None) is KernelRegistry.select:  # another rule is asked every time
            if len(self._call_kernels) >= 4096:
                self._call_kernels = {}
            self._call_kernels[request] = chosen
        return chosen

    def call_kernel(self, kernel: KernelMetadata, *, m: int, n: int, k: int) -> KernelMetadata:
        """The kernel that a whole call runs where select() picked `kernel`.

        select() keeps the FP6 entries for every shape they accept, since the
        separate conversion needs them, and the skinny entry of a single
        height for the M of that height.  A whole call is free to take any
        entry with the same results: of the skinny entries the one that plans
        its rows, and where an FP6 entry fits the smallest predicted time of
        the entries with its operand alignment (kernel_table.predicted_us),
        since on few tiles of 256 rows another one is faster (512 x 4096 x
        4096: FP6 36.7 us, skinny 16.6; 512 x 16384 x 4096: FP6 47.4, FP6_EDGE
        41.9; groups of 128, 128 x 1024 x 4096: FP6 37.8, skinny 12.7).
        Kernels with a figure of the caller's own (with_status) stay."""
        desc = None if kernel.table_index is None else kt.TABLE[kernel.table_index]
        fp6 = desc is not None and desc.operand_format == kt.OPERANDS_FP6
        if not (fp6 or (desc is not None and desc.is_stream and not desc.plans_rows)):
            return kernel
        if kernel.tile.split_k != 1 or kernel.measured_tops != kt.measured_tops(desc):  # as _Candidate.table_figure
            return kernel
        chosen = kernel
        sub = kernel.scale.subchannel_size
        best = kt.predicted_us(desc, m, n, k, sub)
        for other in self._family(kernel.a_dtype, kernel.scale, kernel.epilogue, kernel.layout, kernel.schedule):
            entry = other.desc
            if entry is None or other.split_k != 1 or (entry.is_stream and not entry.plans_rows):
                continue
            if not fp6:
                if entry.plans_rows:
                    return other.kernel
                continue
            if best is None or entry.operand_format == kt.OPERANDS_PACKED or not other.accepts(m, n, k):
                continue
            us = kt.predicted_us(entry, m, n, k, sub)
            if us is not None and us < best:
                chosen, best = other.kernel, us
        return chosen

    def select_reference(
        self,
        *,
        dtype: OperandDType,
        scale: ScaleSpec,
        epilogue: Epilogue,
        layout: GemmLayout = GemmLayout.NN,
        split_k: int | None = 1,
        schedule: KernelSchedule = KernelSchedule.STANDARD,
    ) -> KernelMetadata:
        candidates = [
            c for c in self._family(dtype, scale, epilogue, layout, schedule) if split_k is None or c.split_k == split_k
        ]
        if not candidates:
            raise LookupError(
                f"no reference kernel metadata for dtype={dtype.value}, scale={scale.label}, "
                f"epilogue={epilogue.value}, layout={layout.value}, schedule={schedule.value}"
            )
        # no shape: rank as for a large M (the skinny subchannel figure applies to few rows only)
        return max(candidates, key=lambda c: _selection_key(c, 1 << 30)).kernel

    def with_status(self, kernel_id: str, status: KernelStatus, **updates: object) -> "KernelRegistry":
        copied = KernelRegistry(self._kernels.values())
        copied._kernels[kernel_id] = replace(copied._kernels[kernel_id], status=status, **updates)
        return copied


default_registry = KernelRegistry(iter_supported_kernel_metadata())
