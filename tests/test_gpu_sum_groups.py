"""The cooperative sum's staged and packed forms at the edges of their stages
(cells shorter and longer than a stage's run, cells off the 4-element grid,
more participants than a stage holds, ragged last workgroups), under every kind
of mode pair: the ones the hardware applies, and the ones it does not."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L
from tiler_amd.realize import realize, route

RE = L.PERMITS_REASSOCIATION
FS, FP, KEEP = L.SUBNORMALS_FLUSH_SIGN, L.SUBNORMALS_FLUSH_POSITIVE, L.SUBNORMALS_PRESERVE

# rows, participants, contributors per cell, rounds, participant major, packed
CASES = [
    (2051, 16, 16, 1, False, True), (2049, 20, 25, 1, False, True), (2050, 100, 20, 1, False, True),
    (2048, 2, 70, 1, False, True), (2048, 1, 5, 1, False, True), (3, 64, 64, 1, False, False),
    (5, 128, 36, 1, False, False), (2, 129, 33, 1, False, False), (2, 640, 9, 1, False, False),
    (2, 700, 6, 1, False, False), (9, 48, 10, 3, True, False), (9, 48, 12, 3, False, False),
    (2060, 40, 12, 2, True, False),
]


@pytest.mark.parametrize("rows,P,c,rounds,major,packed", CASES)
def test_form_choice(rows, P, c, rounds, major, packed):
    flags = L.REGION_ALIGNED16 | (L.REGION_PARTICIPANT_MAJOR if major else 0)
    for modes, sfx in (((KEEP, KEEP), ""), ((FS, FS), "_m")):
        rz = realize(L.PROGRAM_SERIAL_SUM, (rows, P * c * rounds), topology=L.SUM_COOPERATIVE,
                     grouping=(P, c, rounds), permissions=RE, flags=flags, input_subnormals=modes[0],
                     result_subnormals=modes[1])
        assert rz.symbols == [f"tiler_sum_f32_cooperative{'_packed' if packed else ''}{sfx}"]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,P,c,rounds,major,packed", CASES)
@pytest.mark.parametrize("modes", [(KEEP, KEEP), (FS, FS), (FS, KEEP), (KEEP, FS), (FP, FS), (FS, FP)])
def test_grouped_sums(ctx, rows, P, c, rounds, major, packed, modes):
    extent = P * c * rounds
    rng = np.random.default_rng(rows * 31 + extent)
    # sums around the subnormal boundary, zeros of both signs, and a few large values
    x = (rng.integers(-2**24, 2**24, (rows, extent)).astype(np.float64) * 2.0**-149).astype(np.float32)
    x[rng.random((rows, extent)) < 0.1] = np.float32(-0.0)
    x[0] = rng.standard_normal(extent).astype(np.float32)
    x[1, extent - 1] = np.nan
    im, rm = modes
    flags = L.REGION_ALIGNED16 | (L.REGION_PARTICIPANT_MAJOR if major else 0)
    rz = realize(L.PROGRAM_SERIAL_SUM, (rows, extent), topology=L.SUM_COOPERATIVE, grouping=(P, c, rounds),
                 permissions=RE, flags=flags, input_subnormals=im, result_subnormals=rm, ctx=ctx)
    dx, do = ctx.to_device(x), ctx.alloc(4 * rows + 4)
    try:
        ctx.fill_u32(do, 0x7FC12345, rows + 1)
        route(ctx, rz, [dx, do])
        got = do.download(np.uint32, (rows + 1,))
    finally:
        dx.free()
        do.free()
    want = oracle.cooperative_grouped_sum(x, rows, extent, P, c, rounds,
                                          layout=oracle.PARTICIPANT_MAJOR if major else oracle.ROUND_MAJOR,
                                          input_mode=im - 1, result_mode=rm - 1)  # the oracle counts modes from 0
    assert np.array_equal(got[:rows], np.ascontiguousarray(want, np.float32).view(np.uint32).reshape(-1))
    assert got[rows] == 0x7FC12345
