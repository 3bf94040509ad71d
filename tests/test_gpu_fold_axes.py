"""Folds whose reduced axes are adjacent, at the edges of their forms: the
column tiles (16 columns, stages of 512 rows, passes of 128), the lane-per-
output batches of 16, and the maximum's row widths, bit for bit with the
oracle's serial fold (tiler-reference/src/evaluate.rs:548-585)."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L
from tiler_amd.realize import realize


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


COLS = [(1, 128, 16), (2, 127, 17), (1, 513, 1), (3, 512, 15), (1, 1025, 33), (2, 640, 271), (17, 130, 2)]
LANES = [(1, 16, 300), (5, 31, 7), (300, 48, 70), (1100, 130, 19), (8192, 128, 2), (1030, 130, 17)]
ROWS = [(1, 16, 1), (70, 256, 1), (1100, 17, 1), (1100, 257, 1), (3, 2049, 1), (1025, 2048, 1)]


@pytest.mark.parametrize("shape,form", [(s, "cols") for s in COLS if s[1] >= 128 and s[2] > 1]
                         + [(s, "lanes") for s in LANES + [s for s in COLS if s[1] < 128]])
@pytest.mark.parametrize("variant,name", [(L.FOLD_SUM, "sum"), (L.FOLD_MAXIMUM, "maximum")])
def test_adjacent_axes_route(shape, form, variant, name):
    rz = realize(L.PROGRAM_FOLD, shape, rank=3, grouping=(0b010,), variant=variant)
    assert rz.symbols == [f"tiler_fold_{name}_f32_{form}"]


@pytest.mark.parametrize("shape,form", [
    # narrow inner axes: the columns' cost is their groups, not their outputs
    ((8192, 128, 2), "lanes"), ((4096, 128, 4), "lanes"), ((2048, 128, 8), "lanes"), ((1024, 128, 3), "cols"),
    ((2048, 4096, 2), "cols"), ((1024, 512, 2), "cols"), ((512, 256, 17), "cols"), ((1024, 256, 17), "lanes"),
    # wide ones: up to one wave of outputs per CU
    ((1, 4096, 4096), "cols"), ((16, 1024, 1024), "cols"), ((1000, 256, 64), "lanes"), ((64, 64, 4096), "lanes"),
])
def test_columns_or_lanes(shape, form):
    rz = realize(L.PROGRAM_FOLD, shape, rank=3, grouping=(0b010,), variant=L.FOLD_SUM)
    assert rz.symbols == [f"tiler_fold_sum_f32_{form}"]


@pytest.mark.parametrize("shape,variant,symbol", [
    ((49152, 21), L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"), ((49153, 21), L.FOLD_MAXIMUM, "tiler_fold_maximum_f32"),
    ((49153, 22), L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"),
    ((262145, 18), L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"),
    ((262145, 17), L.FOLD_MAXIMUM, "tiler_fold_maximum_f32"),
    ((131072, 17), L.FOLD_FMA, "tiler_fold_fma_f32"), ((131073, 17), L.FOLD_FMA, "tiler_sum_f32_staged_r256_u_m"),
    ((65536, 23), L.FOLD_FMA, "tiler_fold_fma_f32"), ((65537, 23), L.FOLD_FMA, "tiler_sum_f32_staged_r256_u_m"),
    ((100, 20), L.FOLD_SQUARED, "tiler_sum_f32_staged_r256_m"), ((100, 17), L.FOLD_SUM, "tiler_sum_f32_staged_r256_u"),
])
def test_short_rows(shape, variant, symbol):
    rz = realize(L.PROGRAM_FOLD, shape, rank=2, grouping=(0b10,), variant=variant, flags=L.REGION_ALIGNED16)
    assert rz.symbols == [symbol]


@pytest.mark.parametrize("shape,mask,symbol", [
    ((4, 8, 64), 0b101, "tiler_fold_sum_f32"),         # not adjacent
    ((2, 5, 300), 0b010, "tiler_fold_sum_f32"),        # too few contributors
    ((4, 2, 64, 8), 0b0101, "tiler_fold_sum_f32"),
    ((4, 1, 64, 8), 0b0101, "tiler_fold_sum_f32_cols"),  # an axis of extent 1 between them moves nothing
    ((4, 1, 64, 8), 0b0110, "tiler_fold_sum_f32_lanes"),
    ((1, 64, 1, 8), 0b0010, "tiler_fold_sum_f32_lanes"),
    ((9, 16, 16), 0b110, "tiler_sum_f32_staged_r1"),   # trailing axes: the staged rows
])
def test_adjacent_axes_are_recognized(shape, mask, symbol):
    rz = realize(L.PROGRAM_FOLD, shape, rank=len(shape), grouping=(mask,))
    assert rz.symbols == [symbol]


@pytest.mark.parametrize("shape,mask,variant,symbol", [
    # 2^32 work items and more do not fit a launch: the grid-stride form takes them
    ((1 << 28, 24), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32"),
    (((1 << 28) - 16, 24), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"),
    ((1 << 26, 257), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32"),
    (((1 << 26) - 4, 257), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"),
    ((1 << 24, 2048), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32"),
    (((1 << 24) - 2, 2048), 0b10, L.FOLD_MAXIMUM, "tiler_fold_maximum_f32_rows"),
    ((1 << 30, 64), 0b10, L.FOLD_SUM, "tiler_fold_sum_f32"),
    (((1 << 30) - 64, 64), 0b10, L.FOLD_SUM, "tiler_sum_f32_staged_r64"),
    ((1 << 30, 64), 0b10, L.FOLD_SQUARED, "tiler_fold_squared_f32"),
    ((1 << 30, 16), 0b10, L.FOLD_SUM, "tiler_sum_f32_staged_r256"),
    ((1 << 16, 16, 1 << 16), 0b010, L.FOLD_SUM, "tiler_fold_sum_f32"),
    ((1 << 16, 16, (1 << 16) - 1), 0b010, L.FOLD_SUM, "tiler_fold_sum_f32_lanes"),
])
def test_launches_stay_within_the_grid(shape, mask, variant, symbol):
    rz = realize(L.PROGRAM_FOLD, shape, rank=len(shape), grouping=(mask,), variant=variant, flags=L.REGION_ALIGNED16)
    assert rz.symbols == [symbol]
    assert all(d.grid[0] * d.block[0] < 1 << 32 for d in rz.dispatches)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", COLS + LANES + ROWS)
@pytest.mark.parametrize("variant", [L.FOLD_SUM, L.FOLD_SQUARED, L.FOLD_FMA, L.FOLD_MAXIMUM])
def test_adjacent_axes_match_the_serial_fold(ctx, shape, variant):
    rng = np.random.default_rng(shape[0] * 7919 + shape[1] * 31 + shape[2] + variant)
    x = (rng.standard_normal(shape) * 3).astype(np.float32)
    flat = x.reshape(-1)
    at = rng.integers(flat.size, size=max(2, flat.size // 97))
    flat[at] = rng.choice(np.array([0.0, -0.0, 1e-40, 3e38, -np.inf, np.nan], np.float32), size=at.size,
                          p=[0.3, 0.3, 0.3, 0.08, 0.01, 0.01])
    x[0, :, 0] = -0.0  # a sum of negative zeros keeps its sign
    sb = (0x40000000, 0x3F800000) if variant == L.FOLD_FMA else (0, 0)
    want = oracle.fold_f32(x, shape, (1,), op=variant, scale_bits=sb[0], bias_bits=sb[1])
    dx, do = ctx.to_device(np.concatenate([np.zeros(1, np.float32), flat])), ctx.alloc(4 * want.size + 8)
    try:
        for off in (0, 4):  # 16-byte aligned storage, then 4-byte
            src = dx.offset(4)
            if off == 0:
                src = ctx.to_device(flat)
            ctx.fill_u32(do, 0x7FC12345, want.size + 2)
            ctx.fold_f32(variant, src, shape, (1,), do.offset(off), scale_bits=sb[0], bias_bits=sb[1])
            ctx.synchronize()
            got = do.download(np.float32, (want.size + 2,))
            assert np.array_equal(bits(got[off // 4:off // 4 + want.size]), bits(want.reshape(-1)))
            assert bits(got)[want.size + off // 4] == 0x7FC12345  # nothing past the outputs
            if off == 0:
                src.free()
    finally:
        dx.free()
        do.free()
