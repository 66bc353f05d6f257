"""Python mirror of the gfx950 kernel table compiled into the library.

The library (csrc/k_dense.hip, csrc/k_ragged.hip) appends its kernels in a
fixed order; this module lists the same entries in the same order so that the
registry can be built without loading the library.  ``native`` checks the
mirror against ``amd_strix_halo_kernels_kernel_table_entry`` the first time it
loads the library and refuses to launch on a mismatch.

This table replaces the reference's tuned gfx1151 tile seeds
(registry.py:112-176) and per-kernel JSON launch metadata.
"""

from __future__ import annotations

import functools
from dataclasses import dataclass

FAMILY_DENSE = 0
FAMILY_RAGGED_FWD = 1
FAMILY_RAGGED_BWD = 2

LAYOUT_NN = 0
LAYOUT_NT = 1
LAYOUT_TN = 2
LAYOUT_TT = 3
LAYOUT_CODES = {"nn": LAYOUT_NN, "nt": LAYOUT_NT, "tn": LAYOUT_TN, "tt": LAYOUT_TT}

SCALE_PER_CHANNEL = 0
SCALE_SUBCHANNEL = 1

EPI_KIND_PLAIN = 0
EPI_KIND_SWIGLU = 2

EPILOGUE_NONE = 0
EPILOGUE_RELU2 = 1
EPILOGUE_SWIGLU = 2

OUT_BF16 = 0
OUT_F32 = 1
OUT_I32 = 2

# Operand formats: PACKED entries read A and B as given; FP6 entries convert
# both int4 operands into a caller workspace in the fp6 (e2m3, v/8) block format
# first (amd_strix_halo_kernels_gemm_workspace_bytes).
OPERANDS_PACKED = 0
OPERANDS_FP6 = 1
# STREAM entries (block_m 16, 32, 64; block_k 32; csrc/shk_skinny.h) read the
# packed operands directly; per-channel calls split a tile's K over several
# workgroups when given a zero-filled workspace (every launch leaves what it
# used zero, counters and partials): sk_split_count / sk_workspace_bytes.
OPERANDS_STREAM = 2
# FP6_EDGE entries run the fp6 tiles on shapes that are no multiple of them:
# the operands are converted with rows padded to 32 and K to 128, and the
# output stops at M and N.
OPERANDS_FP6_EDGE = 3
FP6_MAX_K = 262144
# Largest K of the fp6 entries (32-bit buffer offsets of a tile's panels);
# per-channel calls with K > FP6_MAX_K run in exact K slices of FP6_MAX_K
# whose int32 sums add into the workspace, except on the persistent tile.
FP6_MAX_K_SLICED = 1 << 24
# Largest K per int32 accumulator of the int8 engines' int4 per-channel
# entries: products are widened x16, so |sum| <= 128 * 128 * K < 2^31 needs
# K < 131072 (K = 131072 overflows when every product is (-8) * (-8)).
INT4_ACC_MAX_K = 131071
# Bytes of the library's static scratch array (SHK_NOALLOC_SCRATCH_BYTES): the
# largest fp6 workspace amd_strix_halo_kernels_launch_gemm_noalloc accepts.
NOALLOC_SCRATCH_BYTES = 128 * 1024 * 1024

# Tile schedules (reference metadata.KernelSchedule): STANDARD launches one
# workgroup per tile, PERSISTENT one per resident slot, striding over tiles.
SCHEDULE_STANDARD = 0
SCHEDULE_PERSISTENT = 1

# Device quantization (amd_strix_halo_kernels_quantize): sources and outputs.
SRC_F32 = 0
SRC_F16 = 1
SRC_BF16 = 2
SRC_I8 = 3
QUANT_CODES = 0
QUANT_PACK_COLS = 1
QUANT_PACK_ROWS = 2


@dataclass(frozen=True)
class KernelDesc:
    """One entry of the library's kernel table (struct shk_kernel_desc)."""

    index: int
    family: int
    dtype_bits: int
    layout: int
    scale_mode: int
    min_subchannel: int
    max_subchannel: int
    epilogue_kind: int
    block_m: int
    block_n: int
    block_k: int
    num_waves: int
    num_stages: int
    lds_bytes: int
    group_size_m: int
    operand_format: int = OPERANDS_PACKED
    schedule: int = SCHEDULE_STANDARD
    split_k: int = 1

    @property
    def needs_workspace(self) -> bool:
        return self.operand_format in (OPERANDS_FP6, OPERANDS_FP6_EDGE)

    @property
    def is_stream(self) -> bool:
        return self.operand_format == OPERANDS_STREAM

    @property
    def plans_rows(self) -> bool:
        """A skinny entry whose tiles' height is picked for each call
        (sk_plan) from any M that is a multiple of 16; group_size_m is the
        most 16-row blocks that a tile joins."""
        return self.is_stream and self.group_size_m > 1

    def workspace_bytes(self, m: int, n: int, k: int) -> int:
        """Bytes of the workspace for shape (m, n, k): fp6 operands (FP6;
        per-channel calls with K > FP6_MAX_K add [m, b_cols] int32 sums), the
        split-K counters and partials (STREAM), 0 for PACKED."""
        return _workspace_bytes(self, m, n, k)

    def _workspace_bytes(self, m: int, n: int, k: int) -> int:
        if self.is_stream:
            return sk_workspace_bytes(self, m, n, k)
        if not self.needs_workspace:
            return 0
        b_cols = 2 * n if self.epilogue_kind == EPI_KIND_SWIGLU else n
        if self.operand_format == OPERANDS_FP6_EDGE:
            kw = -(-k // 128) * 128
            return ((-(-m // 32) + -(-b_cols // 32)) * 32 * kw * 3) // 4
        nbytes = (m * k * 3) // 4 + (b_cols * k * 3) // 4
        if self.scale_mode == SCALE_PER_CHANNEL and k > FP6_MAX_K:
            nbytes += 4 * m * b_cols
        return nbytes

    @property
    def max_k(self) -> int | None:
        """Largest logical K a dense entry runs (None: no bound), as the
        library checks it (capi.hip dense_max_k)."""
        if self.family != FAMILY_DENSE:
            return None
        if self.is_stream:
            return FP6_MAX_K_SLICED if (self.dtype_bits == 4 and self.scale_mode == SCALE_PER_CHANNEL) else None
        if self.operand_format == OPERANDS_FP6_EDGE:
            return FP6_MAX_K
        if self.operand_format == OPERANDS_FP6:
            if self.scale_mode == SCALE_PER_CHANNEL and self.schedule == SCHEDULE_PERSISTENT:
                return FP6_MAX_K
            return FP6_MAX_K_SLICED
        if self.dtype_bits == 4 and self.scale_mode == SCALE_PER_CHANNEL:
            return INT4_ACC_MAX_K * max(1, self.split_k)
        return None

    def supports_k(self, k: int) -> bool:
        bound = self.max_k
        return bound is None or k <= bound

    def ragged_workspace_bytes(self, m: int, n: int, k_packed: int, groups: int) -> int:
        """Bytes of the operand workspace of a ragged call (0 for PACKED):
        with K rounded up to 128 (256 for the subchannel entries), the
        forward holds A (round32(m) rows) and per group B (round32(n) rows);
        the backward per group A, then per group B (k_f6ragged.hip)."""
        if not self.needs_workspace or m == 0 or n == 0 or groups == 0:
            return 0
        step = 256 if self.scale_mode == SCALE_SUBCHANNEL else 128
        kw = -(-2 * k_packed // step) * step
        m32, n32 = -(-m // 32) * 32, -(-n // 32) * 32
        if self.family == FAMILY_RAGGED_FWD:
            return (m32 * kw * 3) // 4 + groups * ((n32 * kw * 3) // 4)
        return groups * ((m32 * kw * 3) // 4 + (n32 * kw * 3) // 4)

    def serves_subchannel(self, size: int | None) -> bool:
        if self.scale_mode == SCALE_PER_CHANNEL:
            return size is None
        return size is not None and self.min_subchannel <= size <= self.max_subchannel


# The 32x32 engines (fp6 per-channel, int8 direct-to-LDS) keep each wave's
# 256 bytes of B scales in LDS past the stage ring (shk_f6.h).
MFMA32_SCALE_BYTES = 4 * 256

# Skinny (STREAM) tiles: 4 waves, wave-private rings of stages of 64 source
# bytes per row (shk_skinny.h); 64 output columns per-channel, 16 subchannel
# (the waves share the columns and take the scale groups in turn).
SK_NW = 4
SK_BN = 64
SK_BN_SUBCH = 16
SK_TARGET_UNITS = 256


def _sk_geometry(r: int, swiglu: bool, subch: bool) -> tuple[int, int]:
    """(ring depth, LDS bytes) of a skinny tile of r rows (SkCfg)."""
    bn = SK_BN_SUBCH if subch else SK_BN
    wcols = 2 * bn if swiglu else bn
    stage = r * 64 + wcols * 64 + ((r // 16) * 256 + 256 if subch else 0)
    tiles = (r // 16) * (wcols // 16)
    ch = (4 if tiles == 1 else 2 if tiles == 2 else 1) if subch else 0  # groups per wave and round
    chain = 2 * SK_NW * ch * tiles * 1024  # two rounds of scaled partials
    budget = 79872 - chain
    depth = 4 if SK_NW * 4 * stage <= budget else (3 if SK_NW * 3 * stage <= budget else 2)
    ring = SK_NW * depth * stage
    red = 0 if subch else SK_NW * (wcols // 16) * 1024
    return depth, max(ring, red) + chain


def _sk_needed_splits(bits: int, k: int) -> int:
    need = 1
    if bits == 4:
        while need * 4 * 1023 < -(-k // 128):
            need *= 2
    return need


def _sk_splits(bits: int, tiles: int, k: int) -> int:
    nst = -(-k // (128 if bits == 4 else 64))
    s = 1
    while s * 2 <= 16 and tiles * s * 2 <= SK_TARGET_UNITS and nst >= 16 * s:
        s *= 2
    return max(s, _sk_needed_splits(bits, k))


# Time fits of the skinny tiles by [8-bit][SwiGLU][16, 32, 64 rows], and for
# subchannel [8-bit][SwiGLU][groups of a stage or more][16, 32 rows]
# (shk_table.h sk_plan, which states the terms).
_SK_FIT = ((((3.76, 2.96, 0.96, 3.11, 0.2, 0.77, 0.1, 1.39, 0.88),
             (3.91, 4.12, 1.8, 2.72, 0.16, 0.54, 0.65, 1.07, 1.19),
             (4.89, 5.84, 2.69, 3.29, 0.33, 1.19, 0.64, 0.1, 1.64)),
            ((3.91, 5.25, 4.09, 1.05, 0.67, 0.92, 0.07, 1.09, 1.19),
             (4.97, 6.96, 6.16, 0.83, 1.12, 0.51, 3.21, 0.32, 1.55),
             (6.94, 9.81, 8.75, 0.0, 0.81, 0.14, 5.91, 1.36, 2.78))),
           (((3.71, 3.68, 4.83, 0.45, 0.0, 0.41, 0.0, 3.55, 1.02),
             (3.64, 5.78, 5.15, 2.5, 0.0, 0.55, 0.0, 3.24, 1.09),
             (4.16, 8.21, 7.34, 4.93, 0.0, 0.77, 0.0, 2.21, 1.59)),
            ((2.87, 10.23, 6.51, 4.32, 1.34, 0.51, 0.0, 3.5, 1.14),
             (3.74, 11.02, 7.83, 4.71, 2.69, 0.0, 2.68, 3.73, 1.71),
             (5.52, 14.08, 12.06, 1.6, 1.05, 0.14, 4.59, 2.99, 2.72))))
_SK_SUB_FIT = (((((3.5, 2.26, 3.42, 2.89, 3.49, 1.45, 0.15, 0.89, 0.44, 0.13),
                  (3.48, 0.06, 6.6, 0.44, 6.75, 1.04, 0.47, 0.98, 0.0, 0.05)),
                 ((3.63, 1.63, 1.64, 2.68, 1.95, 0.89, 0.77, 0.72, 1.53, 0.6),
                  (3.84, 4.06, 3.62, 4.79, 3.72, 1.07, 0.55, 1.02, 0.79, 0.37))),
                (((3.84, 0.47, 6.04, 0.29, 6.52, 0.39, 0.71, 1.01, 0.96, 0.62),
                  (3.78, 0.14, 10.11, 0.68, 10.49, 0.0, 1.15, 1.06, 0.74, 0.64)),
                 ((4.0, 3.09, 4.1, 5.12, 3.22, 1.21, 0.64, 0.97, 2.21, 1.16),
                  (3.86, 4.44, 6.46, 6.36, 5.75, 2.24, 0.0, 1.03, 1.13, 0.8)))),
               ((((3.59, 0.0, 3.86, 0.0, 4.24, 0.0, 0.56, 0.91, 1.52, 0.59),
                  (3.41, 0.0, 5.68, 0.0, 6.02, 0.0, 0.84, 0.94, 1.15, 0.48)),
                 ((3.42, 2.59, 1.44, 4.91, 1.73, 1.86, 0.55, 0.57, 4.23, 1.94),
                  (3.84, 5.39, 3.26, 9.06, 2.89, 2.21, 0.0, 0.84, 2.47, 1.64))),
                (((3.86, 0.0, 5.44, 0.0, 5.84, 0.0, 0.82, 1.02, 2.57, 0.75),
                  (3.38, 0.0, 9.69, 0.0, 10.3, 0.0, 1.15, 0.91, 3.97, 1.54)),
                 ((3.9, 4.15, 2.68, 9.52, 1.89, 2.21, 1.68, 0.63, 6.05, 4.11),
                  (3.31, 6.32, 6.61, 11.59, 3.82, 2.14, 0.0, 0.74, 5.02, 3.92)))))


@functools.lru_cache(maxsize=4096)
def sk_plan(bits: int, sub: int, swiglu: bool, m: int, n: int, k: int, layout: int = LAYOUT_NN) -> tuple[int, float]:
    """(tile rows, predicted us) of a call of M rows on a skinny entry that
    plans its rows (shk_table.h sk_plan, which states the fits); sub: the
    group size, 0 for per-channel scales."""
    best, whole = (16, -1.0), (16, -1.0)
    for i in range(2 if sub else 3):
        rows = 16 << i
        if i > 0 and m <= rows // 2:
            break
        if not sub and m % rows and _sk_needed_splits(bits, k) > 1:
            continue
        tiles = -(-m // rows) * (n // (SK_BN_SUBCH if sub else SK_BN))
        s = 1 if sub else _sk_splits(bits, tiles, k)
        u = tiles * s
        w = k / s / 4096.0
        second = u > 256
        past = u / 256.0 - 1.0 if second else 0.0
        wm, w2, twice = w * (1.0 + past), w if second else 0.0, (u - 1) // 512
        a_mn, b_mn = wm if layout == LAYOUT_TN else 0.0, wm if layout == LAYOUT_NN else 0.0
        if sub:
            g = k / sub / 32.0
            fit = _SK_SUB_FIT[bits == 8][swiglu][sub >= (128 if bits == 4 else 64)][i]
            terms = (1.0, w, g, w * twice, g * twice, w2, g if second else 0.0, past, a_mn, b_mn)
        else:
            fit = _SK_FIT[bits == 8][swiglu][i]
            rounds = (u - 1) // 256
            terms = (1.0, w, w * rounds, w * twice, w2, past, float(rounds), a_mn, float(s.bit_length() - 1))
        us = 0.0
        for f, x in zip(fit, terms):
            us += f * x
        if best[1] < 0.0 or us < best[1]:
            best = (rows, us)
        if m % rows == 0:
            whole = (rows, us)
    return whole if whole[1] <= 1.05 * best[1] else best


def _sk_tile_rows(desc: "KernelDesc", m: int, n: int, k: int) -> int:
    """Rows of a skinny entry's tiles."""
    if not desc.plans_rows:
        return desc.block_m
    return sk_plan(desc.dtype_bits, 0, desc.epilogue_kind == EPI_KIND_SWIGLU, m, n, k, desc.layout)[0]


def sk_split_count(desc: "KernelDesc", m: int, n: int, k: int, with_workspace: bool = True) -> int:
    """Workgroups sharing a skinny per-channel tile's K (shk_table.h
    sk_splits): about SK_TARGET_UNITS workgroups with at least two
    stages per wave, at most 16; for int4 enough to keep every wave within
    1023 stages of 128 K.  Without a workspace 1, or 0 if K needs a split."""
    if desc.scale_mode == SCALE_SUBCHANNEL:
        return 1
    if not with_workspace:
        return 1 if _sk_needed_splits(desc.dtype_bits, k) == 1 else 0
    rows = _sk_tile_rows(desc, m, n, k)
    return _sk_splits(desc.dtype_bits, -(-m // rows) * (n // desc.block_n), k)


def sk_workspace_bytes(desc: "KernelDesc", m: int, n: int, k: int) -> int:
    """Arrival counters (padded to 256 bytes) and exact int32 partials of a
    split skinny launch; 0 when it runs unsplit (shk_table.h)."""
    s = sk_split_count(desc, m, n, k, True)
    if s <= 1:
        return 0
    rows = _sk_tile_rows(desc, m, n, k)
    tiles = -(-m // rows) * (n // desc.block_n)
    cf = 2 if desc.epilogue_kind == EPI_KIND_SWIGLU else 1
    return ((tiles * 4 + 255) & ~255) + tiles * s * (desc.block_n // 16) * (rows // 16) * cf * 1024


def _desc(index, family, bits, layout, *, bm, bn, bk, wm, wn, swiglu=False, subch=False, mk=64, group_m=8, pipe=0,
          fp6=False, fp6_sub=False, fp6_small=False, schedule=SCHEDULE_STANDARD, split_k=1):
    # pipe > 0: direct-to-LDS engine with a ring of `pipe` packed stages of 64
    # source bytes per tile row; 0: register-staged engine, two widened stages.
    # fp6: three stages of 256 A rows + 256 B rows x 128 K in fp6 (96 bytes).
    # fp6_sub: a 72 KiB ring of 128 + 128 rows in fp6 (96 bytes per 128 K) and
    # an eight-slot scale ring (shk_f6sub.h).  Groups of 256 run three 128-K
    # stage slots (the entry's num_stages, 3) and four 768-byte scale slots;
    # groups of 64 and 128 run six 64-K slots of the same ring, one or two per
    # group, and eight 768-byte scale slots; groups of 32 two per 64-K slot and
    # eight 1024-byte scale slots (two b_scale rows each), the entry's LDS.
    # fp6_small: two stages of 128 A rows + 128 B rows x 128 K in fp6 (96
    # bytes), then the B-scale slots (shk_f6small.h; k_f6ragged.hip).
    brows = 2 * bn if swiglu else bn
    if fp6_small:
        fp6 = True
        pipe = 2
        lds = pipe * (bm + bn) * 96 + MFMA32_SCALE_BYTES
    elif fp6_sub:
        fp6 = True
        pipe = 3
        lds = pipe * (bm + bn) * 96 + 8 * 1024
    elif fp6:
        pipe = 3
        lds = pipe * (bm + 256) * 96 + MFMA32_SCALE_BYTES
    else:
        lds = pipe * (bm + brows) * 64 if pipe else 2 * (bm * bk + brows * bk)
        if bits == 8 and pipe:
            lds += MFMA32_SCALE_BYTES
    return KernelDesc(
        index=index,
        family=family,
        dtype_bits=bits,
        layout=layout,
        scale_mode=SCALE_SUBCHANNEL if subch else SCALE_PER_CHANNEL,
        min_subchannel=(32 if mk == 32 or fp6_sub else 64) if subch else 0,
        max_subchannel=(32 if mk == 32 else 256) if subch else 0,
        epilogue_kind=EPI_KIND_SWIGLU if swiglu else EPI_KIND_PLAIN,
        block_m=bm,
        block_n=bn,
        block_k=bk,
        num_waves=wm * wn,
        num_stages=pipe or 2,
        lds_bytes=lds,
        group_size_m=group_m,
        operand_format=OPERANDS_FP6 if fp6 else OPERANDS_PACKED,
        schedule=schedule,
        split_k=split_k,
    )


def _sk_desc(index, bits, layout, r, *, swiglu=False, subch=False, schedule=SCHEDULE_STANDARD, split_k=1):
    depth, lds = _sk_geometry(r, swiglu, subch)
    return KernelDesc(
        index=index, family=FAMILY_DENSE, dtype_bits=bits, layout=layout,
        scale_mode=SCALE_SUBCHANNEL if subch else SCALE_PER_CHANNEL,
        min_subchannel=32 if subch else 0, max_subchannel=256 if subch else 0,
        epilogue_kind=EPI_KIND_SWIGLU if swiglu else EPI_KIND_PLAIN,
        block_m=r, block_n=SK_BN_SUBCH if subch else SK_BN, block_k=32, num_waves=SK_NW, num_stages=depth,
        lds_bytes=lds,
        group_size_m=1, operand_format=OPERANDS_STREAM, schedule=schedule, split_k=split_k)


def _sk_rows_desc(index, bits, layout, *, swiglu, subch):
    # the figures of the tallest tile
    r = 32 if subch else 64
    depth, lds = _sk_geometry(r, swiglu, subch)
    return KernelDesc(
        index=index, family=FAMILY_DENSE, dtype_bits=bits, layout=layout,
        scale_mode=SCALE_SUBCHANNEL if subch else SCALE_PER_CHANNEL,
        min_subchannel=32 if subch else 0, max_subchannel=256 if subch else 0,
        epilogue_kind=EPI_KIND_SWIGLU if swiglu else EPI_KIND_PLAIN, block_m=16,
        block_n=SK_BN_SUBCH if subch else SK_BN, block_k=32, num_waves=SK_NW, num_stages=depth, lds_bytes=lds,
        group_size_m=r // 16, operand_format=OPERANDS_STREAM)


def _edge_desc(index, layout, bm, *, swiglu=False, subch=False):
    # the ring of the largest kernel the entry may launch (the 256-row
    # per-channel tile, the subchannel tile; _desc), at its granularity
    return KernelDesc(
        index=index, family=FAMILY_DENSE, dtype_bits=4, layout=layout,
        scale_mode=SCALE_SUBCHANNEL if subch else SCALE_PER_CHANNEL, min_subchannel=32 if subch else 0,
        max_subchannel=256 if subch else 0, epilogue_kind=EPI_KIND_SWIGLU if swiglu else EPI_KIND_PLAIN,
        block_m=bm, block_n=64, block_k=64 if subch else 32, num_waves=4, num_stages=3,
        lds_bytes=3 * (128 + 128) * 96 + 8 * 1024 if subch else 3 * (256 + 256) * 96 + MFMA32_SCALE_BYTES,
        group_size_m=8, operand_format=OPERANDS_FP6_EDGE)


def _build() -> tuple[KernelDesc, ...]:
    out: list[KernelDesc] = []

    def add(**kw):
        out.append(_desc(len(out), **kw))

    def add_sk(*args, **kw):
        out.append(_sk_desc(len(out), *args, **kw))

    for bits in (4, 8):
        big_bk = 128 if bits == 4 else 64
        for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
            d = dict(family=FAMILY_DENSE, bits=bits, layout=layout)
            if bits == 4:
                add(**d, bm=256, bn=256, bk=128, wm=2, wn=2, fp6=True)
                add(**d, bm=256, bn=128, bk=128, wm=2, wn=2, swiglu=True, fp6=True)
                add(**d, bm=128, bn=128, bk=128, wm=2, wn=2, subch=True, fp6_sub=True)
            add(**d, bm=256, bn=256, bk=big_bk, wm=2, wn=2, pipe=4)
            add(**d, bm=256, bn=128, bk=big_bk, wm=2, wn=2, swiglu=True, pipe=4)
            add(**d, bm=128, bn=128, bk=64, wm=2, wn=2)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, swiglu=True)
            add(**d, bm=256, bn=128, bk=big_bk, wm=4, wn=2, subch=True)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, subch=True)
            add(**d, bm=256, bn=64, bk=big_bk, wm=4, wn=2, swiglu=True, subch=True)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, swiglu=True, subch=True)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, subch=True, mk=32)
            add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, swiglu=True, subch=True, mk=32)
    for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN, LAYOUT_TT):
        # fp6 entries lead each family (k_ragged.hip)
        add(family=FAMILY_RAGGED_FWD, bits=4, layout=layout, group_m=1, bm=128, bn=128, bk=128, wm=2, wn=2,
            fp6_small=True)
        add(family=FAMILY_RAGGED_FWD, bits=4, layout=layout, group_m=1, bm=128, bn=128, bk=128, wm=2, wn=2,
            subch=True, fp6_sub=True)
        for subch, mk in ((False, 64), (True, 64), (True, 32)):
            f = dict(family=FAMILY_RAGGED_FWD, bits=4, layout=layout, subch=subch, mk=mk, group_m=1)
            add(**f, bm=16, bn=128, bk=128, wm=1, wn=4)
            add(**f, bm=32, bn=128, bk=128, wm=2, wn=2)
            add(**f, bm=64, bn=128, bk=128, wm=2, wn=2)
            add(**f, bm=128, bn=128, bk=128, wm=2, wn=2)
        add(family=FAMILY_RAGGED_BWD, bits=4, layout=layout, group_m=1, bm=128, bn=128, bk=128, wm=2, wn=2,
            fp6_small=True)
        add(family=FAMILY_RAGGED_BWD, bits=4, layout=layout, group_m=1, bm=128, bn=128, bk=128, wm=2, wn=2,
            subch=True, fp6_sub=True)
        for subch, mk in ((False, 64), (True, 64), (True, 32)):
            add(family=FAMILY_RAGGED_BWD, bits=4, layout=layout, subch=subch, mk=mk, group_m=1, bm=128, bn=128,
                bk=128, wm=2, wn=2)
    # persistent int4 entries (plain epilogue kind) after the ragged families
    for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
        d = dict(family=FAMILY_DENSE, bits=4, layout=layout, schedule=SCHEDULE_PERSISTENT)
        add(**d, bm=256, bn=256, bk=128, wm=2, wn=2, fp6=True)
        add(**d, bm=128, bn=128, bk=128, wm=2, wn=2, subch=True, fp6_sub=True)
        add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, subch=True)
        add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, subch=True, mk=32)
    # split-K 2/4/8 (fp32 output): 128x128 per-channel, int4 64x64 subchannel
    for bits in (4, 8):
        for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
            d = dict(family=FAMILY_DENSE, bits=bits, layout=layout)
            for split in (2, 4, 8):
                add(**d, bm=128, bn=128, bk=64, wm=2, wn=2, split_k=split)
            if bits == 4:
                for mk in (64, 32):
                    for split in (2, 4, 8):
                        add(**d, bm=64, bn=64, bk=64, wm=2, wn=2, subch=True, mk=mk, split_k=split)
    # skinny tiles (k_skinny.hip), per (bits, layout)
    for bits in (4, 8):
        for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
            for r in (16, 32, 64):
                for swiglu, subch in ((False, False), (True, False), (False, True), (True, True)):
                    add_sk(bits, layout, r, swiglu=swiglu, subch=subch)
            if bits == 4:
                for split in (1, 2, 4, 8):
                    for r in (16, 32, 64):
                        for subch in (False, True):
                            add_sk(bits, layout, r, subch=subch, schedule=SCHEDULE_PERSISTENT, split_k=split)
            for split in (2, 4, 8):
                for r in (16, 32, 64):
                    for subch in (False, True):
                        add_sk(bits, layout, r, subch=subch, split_k=split)
    # fp6 entries for shapes that are no tile multiples (k_f6edge.hip)
    for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
        for bm in (64, 16):
            for subch in (False, True):
                for swiglu in (False, True):
                    out.append(_edge_desc(len(out), layout, bm, swiglu=swiglu, subch=subch))
    # skinny entries that plan their rows (k_skinny.hip sk_rows_entry)
    for bits in (4, 8):
        for layout in (LAYOUT_NN, LAYOUT_NT, LAYOUT_TN):
            for subch in (False, True):
                for swiglu in (False, True):
                    out.append(_sk_rows_desc(len(out), bits, layout, swiglu=swiglu, subch=subch))
    return tuple(out)


TABLE: tuple[KernelDesc, ...] = _build()


@functools.lru_cache(maxsize=4096)
def _workspace_bytes(desc: KernelDesc, m: int, n: int, k: int) -> int:
    # memoized: mm() sizes the workspace on every call
    return desc._workspace_bytes(m, n, k)


def measured_tops(desc: KernelDesc) -> float | None:
    """Throughput measured on MI355X (bench.py and sweeps on one GPU; the
    whole call including operand conversion), used by the registry's
    selection like the reference's benchmark TOPS (registry.py:254-352):
    fp6 int4 per-channel 256x256 (C2, 8192^3), fp6 int4 SwiGLU 256x128
    (4096 x 2*11008 x 4096), fp6 int4 subchannel 128x128 (C3), int8 32x32
    SwiGLU 256x128 (C4) and int8 plain 256x256 (8192^3), and the skinny
    tiles (SKINNY_TOPS, SKINNY_SUB_TOPS).  Other entries have no measurement
    and rank by tile area."""
    if desc.family != FAMILY_DENSE or desc.schedule != SCHEDULE_STANDARD or desc.split_k > 1:
        return None
    if desc.operand_format == OPERANDS_FP6:
        if desc.scale_mode == SCALE_SUBCHANNEL:
            return 2001.0
        return 3504.0 if desc.epilogue_kind == EPI_KIND_PLAIN else 3161.0
    if desc.operand_format == OPERANDS_STREAM:
        if desc.scale_mode == SCALE_PER_CHANNEL:
            return SKINNY_TOPS
        return SKINNY_SUB_TOPS[32 if desc.plans_rows else desc.block_m]
    if desc.dtype_bits == 8 and desc.num_stages == 4 and desc.block_m == 256:
        return 2014.0 if desc.epilogue_kind == EPI_KIND_SWIGLU else 2270.0
    return None


# The skinny per-channel tiles' figure: the bench's skinny line (int4, M = 16,
# N = K = 8192, 8.9 us per launch: 241 TOPS).  int8 and SwiGLU skinny tiles
# carry it too: at N = K = 4096 and M = 64 to 4160 every skinny per-channel
# tile (int4 and int8, plain and SwiGLU) ran 1.2-3x faster than the
# register-staged 64x64 and 128x128 tiles, which outranked it by area.  The
# larger measured tiles keep their higher figures where they fit.
SKINNY_TOPS = 241.0

# The skinny subchannel tiles' figures by tile height: int4, N = K = 8192,
# groups of 128; 16 rows at M = 16 (22.3 us, 96 TOPS), 32 and 64 rows at
# M = 64 (46.6 and 56.6 us: 184 and 152 TOPS), so the 32-row tile, the
# fastest of them at M = 64 and 192, ranks first where it fits.  They rank
# above the register-staged subchannel tiles up to M = SKINNY_SUB_MAX_M rows:
# at N = K = 4096 they ran 3x faster at M = 64 and 1.0-1.4x at M = 192, and
# from M = 576 up to 1.8x slower (groups of 32 from M = 320).
SKINNY_SUB_TOPS = {16: 96.0, 32: 184.0, 64: 152.0}
SKINNY_SUB_MAX_M = 256


# CUs of an MI355X: a round of one workgroup each (shk_table.h kF6EdgeCus).
_CUS = 256


def _f6_edge_us(m: int, n: int, k: int, swiglu: bool) -> float:
    """GEMM time (us) of an FP6_EDGE per-channel call as the launcher splits
    it (shk_table.h f6_edge_plan): 256-row tiles, half-height ones in a
    partial last round that holds them, or 128 x 128 tiles."""
    k1 = k / 1024.0
    bn = 128 if swiglu else 256
    tm, tn, tm2 = -(-m // 256), -(-n // bn), -(-m // 128)
    rounds, rest = divmod(tm * tn, _CUS)
    round_us = 14.0 + 4.9 * k1
    us = round_us * (rounds + (1 if rest else 0))
    if rest:
        c = tn if rounds == 0 else -(-rest // tm)
        if tm2 * c <= _CUS:
            us = round_us * (rounds + 0.6)
    if not swiglu:
        small = (2.6 + 2.05 * k1) * -(-(tm2 * -(-n // 128)) // _CUS)
        us = min(us, small)
    return us


PREDICT_MAX_K = 65536  # K up to which the fits of predicted_us stand

# subchannel: a 128 x 128 fp6 tile's fixed us and us per K value by group
# size; the 64 x 64 tile's us by [SwiGLU][NN, NT, TN] for a round of 256 tiles
# (constant, K / 1024, K / 8 groups) and for the tiles past it (the same)
_PACKED_SUB_US = (
    ((3.18, 9.2, 3.26, 2.83, 1.36, 0.9), (2.93, 4.84, 3.42, 1.47, 1.31, 0.83), (3.4, 12.61, 3.5, 4.53, 2.14, 1.09)),
    ((2.87, 11.52, 5.56, 7.46, 3.23, 0.79), (3.64, 7.13, 5.28, 1.63, 3.65, 1.59), (3.4, 15.99, 5.23, 0.0, 5.86, 0.0)),
)
_F6_SUB_US = {32: (5.0, 0.0215), 64: (5.0, 0.0125), 128: (5.0, 0.0061), 256: (3.5, 0.0038)}


def predicted_us(desc: KernelDesc, m: int, n: int, k: int, sub: int | None = None) -> float | None:
    """Predicted time of a standard int4 call on an entry, in us (None for the
    other families and K past PREDICT_MAX_K); capi.hip computes the skinny,
    FP6_EDGE and 64 x 64 entries' alike, and the skinny entries of a family
    share the planned tiles' time (among them selection_area decides):

    * skinny tiles: sk_plan;
    * the subchannel 64 x 64 tile on the packed operands, past
      SKINNY_SUB_MAX_M rows (below them the skinny tiles' figures stand):
      linear in K, groups and tiles past a round, by layout;
    * fp6 entries: two launches, the conversion at 5 TB/s, then rounds of
      tiles: per-channel 256-row tiles (FP6) or the launcher's split
      (FP6_EDGE); subchannel 128 x 128 tiles, two a CU (1.3 times one; 1.1
      beside half-height tiles, which alone take 0.8).

    Fitted to calls drawn over M 16..8192, N 512..16384 and K 512..14336 in
    every layout, each entry measured (us): the predicted choice takes 1.2%
    (per-channel), 0.6% (subchannel) and 0.8, 0.4% (SwiGLU) more than the best
    of the entries, and of 5200 calls 23 take 3% more than on the entry that
    the figures alone, without predictions, rank first.  Groups of 64, 1536 x
    704 x 768 NT: 64 x 64 tile 12.4, edge 18.1, skinny 24.6; groups of 128, 320
    x 16384 x 4096 skinny 221, edge 56.5; per-channel 8176 x 16384 x 4096
    skinny 810, edge 324."""
    if (desc.family != FAMILY_DENSE or desc.dtype_bits != 4 or desc.schedule != SCHEDULE_STANDARD
            or desc.split_k > 1 or k > PREDICT_MAX_K):
        return None
    swiglu = desc.epilogue_kind == EPI_KIND_SWIGLU
    cols = 2 * n if swiglu else n
    convert = 6.0 + 2.5e-7 * ((m + cols) * k)
    if desc.scale_mode == SCALE_SUBCHANNEL:
        if sub not in _F6_SUB_US:
            return None
        if desc.is_stream:
            # of the heights, the 32-row tile ranks first, as measured (SKINNY_SUB_TOPS)
            rank = 1.0 if desc.plans_rows else {32: 1.0, 64: 1.001, 16: 1.002}[desc.block_m]
            return rank * sk_plan(4, sub, swiglu, m, n, k, desc.layout)[1]
        if desc.operand_format == OPERANDS_PACKED:
            if desc.block_m != 64 or desc.block_n != 64 or m <= SKINNY_SUB_MAX_M:
                return None
            u = float((m // 64) * (n // 64))
            past = u / 256.0 - 1.0 if u > 256.0 else 0.0
            w, g = k / 1024.0, k / sub / 8.0
            us = 0.0
            for f, x in zip(_PACKED_SUB_US[swiglu][desc.layout], (1.0, w, g, w * past, g * past, past)):
                us += f * x
            return us
        if not desc.needs_workspace:
            return None
        fixed, per_k = _F6_SUB_US[sub]
        columns = -(-n // 64) if swiglu else -(-n // 128)
        whole, tiles = (m + 63) // 128 * columns, -(-m // 128) * columns  # the others half as high
        rounds = 1.0
        if tiles > _CUS:
            rounds = 1.1 if whole <= _CUS and tiles <= 2 * _CUS else 1.3 * -(-(whole + tiles) // (4 * _CUS))
        if whole == 0:
            rounds *= 0.8
        return convert + (fixed + per_k * k) * rounds
    if desc.operand_format == OPERANDS_STREAM:
        return sk_plan(4, 0, swiglu, m, n, k, desc.layout)[1]
    if desc.operand_format == OPERANDS_FP6_EDGE:
        return convert + _f6_edge_us(m, n, k, swiglu)
    if desc.operand_format == OPERANDS_FP6:
        tiles = (m // desc.block_m) * (n // desc.block_n)
        return convert + (14.0 + 4.9 * (k / 1024.0)) * -(-tiles // _CUS)
    return None


def selection_tops(desc: KernelDesc, m: int, n: int | None = None, k: int | None = None,
                   sub: int | None = None) -> float | None:
    """The throughput by which select ranks an entry for a shape (capi.hip
    measured_score): an int4 skinny or FP6_EDGE entry's predicted one, below
    the FP6 entries' figures (a caller of the separate conversion needs an
    FP6 entry where one fits); for the others, or without n and k,
    measured_tops, where the skinny subchannel tiles' figure holds up to
    SKINNY_SUB_MAX_M rows."""
    if n is not None and k is not None and desc.dtype_bits == 4 and desc.operand_format != OPERANDS_FP6:
        us = predicted_us(desc, m, n, k, sub)
        if us is not None:
            cap = 2000.0 if desc.scale_mode == SCALE_SUBCHANNEL else 3000.0
            return min(cap, 2.0 * float(m) * float(n) * float(k) / us / 1e6)
    tops = measured_tops(desc)
    if (tops is not None and desc.operand_format == OPERANDS_STREAM and desc.scale_mode == SCALE_SUBCHANNEL
            and m > SKINNY_SUB_MAX_M):
        return None
    return tops


def selection_area(desc: KernelDesc, m: int) -> int:
    """The second ranking key of select for M rows, a tile's area (capi.hip
    selection_area).  A skinny entry that plans its rows counts as a 16-row
    tile, just before the entry of that height; subchannel calls past
    SKINNY_SUB_MAX_M rows find it before every skinny entry of one height."""
    if desc.plans_rows:
        tall = desc.scale_mode == SCALE_SUBCHANNEL and m > SKINNY_SUB_MAX_M
        return (64 if tall else 16) * desc.block_n + 1
    return desc.block_m * desc.block_n


def entries(family: int) -> tuple[KernelDesc, ...]:
    return tuple(d for d in TABLE if d.family == family)


@functools.lru_cache(maxsize=None)
def ragged_task_capacity(rows: int, groups: int, tile: int) -> int:
    """Upper bound on the row tasks of `rows` rows in `groups` groups with
    tasks of `tile` rows (amd_strix_halo_kernels_ragged_task_capacity): every
    group adds at most one partial task at each end."""
    if rows < 0 or groups < 0 or tile <= 0:
        return 0
    return min(rows // tile + 2 * groups + 1, 0x7FFFFFFF)


@functools.lru_cache(maxsize=None)
def find_ragged(family: int, *, layout: int, subchannel: int | None, block_m: int | None = None,
                fp6: bool = False) -> KernelDesc:
    """Ragged kernel for a layout and scale mode (and task rows for the
    forward): an FP6 entry if `fp6`, else one that reads the packed operands."""
    fmt = OPERANDS_FP6 if fp6 else OPERANDS_PACKED
    for d in TABLE:
        if d.family != family or d.layout != layout or not d.serves_subchannel(subchannel):
            continue
        if d.operand_format != fmt:
            continue
        if block_m is not None and d.block_m != block_m:
            continue
        return d
    raise LookupError(
        f"no gfx950 ragged kernel for family={family}, layout={layout}, subchannel={subchannel}, block_m={block_m}, "
        f"fp6={fp6}"
    )


def ragged_fp6_eligible(family: int, *, subchannel: int | None, m: int, n: int, k_packed: int) -> bool:
    """Whether a ragged call's sizes suit the fp6 entries (k_f6ragged.hip):
    N a multiple of 8 (whole 16-byte output units) and K at most FP6_MAX_K;
    per-channel, or subchannel with M * ceil(K/S) even (the tile reads
    a_scale in whole dwords; groups of 32 in pairs, so ceil(K/32) even)."""
    if subchannel is not None:
        cols = -(-2 * k_packed // subchannel)
        if m * cols % 2 or (subchannel == 32 and cols % 2):
            return False
    return n % 8 == 0 and 2 * k_packed <= FP6_MAX_K


# Task rows of the forward kernels that read packed operands, and of the fp6
# forward (whose task list is built with align_tile 32).
RAGGED_FWD_BLOCK_M = tuple(sorted({d.block_m for d in entries(FAMILY_RAGGED_FWD) if not d.needs_workspace}))
RAGGED_FP6_BLOCK_M = 128
# RaggedDotConfig.block_m that asks for the fp6 forward (as does the default,
# 64, where the fp6 kernel applies); the other heights pick the packed kernels.
RAGGED_FP6_CONFIG_BLOCK_M = 256
RAGGED_FP6_ALIGN = 32
