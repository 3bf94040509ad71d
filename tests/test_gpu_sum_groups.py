"""The cooperative sum's direct, staged and packed forms at the edges of their
stages (cells shorter and longer than a stage's run, cells off the 4-element
grid, more participants than a stage holds, ragged last workgroups) and of the
rule that chooses between them, under every kind of mode pair: none, the ones
the hardware applies, and the ones it does not."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L
from tiler_amd.realize import realize, route

RE = L.PERMITS_REASSOCIATION
FS, FP, KEEP = L.SUBNORMALS_FLUSH_SIGN, L.SUBNORMALS_FLUSH_POSITIVE, L.SUBNORMALS_PRESERVE

# rows, participants, contributors per cell, rounds, participant major, and the
# form (direct, staged, packed) without modes, under the hardware's, under others
CASES = [
    (2051, 16, 16, 1, False, "ppp"), (2049, 20, 25, 1, False, "ppp"), (2050, 100, 20, 1, False, "ppd"),
    (2048, 2, 70, 1, False, "ppp"), (2048, 1, 5, 1, False, "ppp"), (3, 64, 64, 1, False, "ssd"),
    (5, 128, 36, 1, False, "dsd"), (2, 129, 33, 1, False, "dsd"), (2, 640, 9, 1, False, "dsd"),
    (2, 700, 6, 1, False, "dsd"), (9, 48, 10, 3, True, "dsd"), (9, 48, 12, 3, False, "dsd"),
    (2060, 40, 12, 2, True, "ddd"),
    (257, 129, 33, 1, False, "sss"), (257, 128, 36, 2, True, "sss"), (256, 700, 66, 1, False, "sss"),
    (2048, 128, 1, 1, False, "dpd"), (2048, 64, 64, 1, False, "ppp"), (2048, 65, 64, 1, False, "pps"),
    (1025, 47, 3, 2, False, "ddd"), (1024, 4, 3, 2, False, "dsd"), (3, 3, 5, 2, True, "ddd"),
    (2, 3, 64, 1, False, "ssd"), (1030, 20, 66, 1, False, "dsd"), (1025, 32, 64, 2, True, "ssd"),
    (300, 50, 65, 2, True, "sss"), (260, 64, 17, 2, True, "sss"), (65536, 4, 4, 2, False, "ddd"),
]
FORMS = {"d": "", "s": "_staged", "p": "_packed"}


@pytest.mark.parametrize("rows,P,c,rounds,major,forms", CASES)
def test_form_choice(rows, P, c, rounds, major, forms):
    flags = L.REGION_ALIGNED16 | (L.REGION_PARTICIPANT_MAJOR if major else 0)
    for modes, form in (((KEEP, KEEP), forms[0]), ((FS, FS), forms[1]), ((FS, KEEP), forms[1]), ((FP, FP), forms[2]),
                        ((KEEP, FS), forms[2]), ((FS, FP), forms[2])):
        rz = realize(L.PROGRAM_SERIAL_SUM, (rows, P * c * rounds), topology=L.SUM_COOPERATIVE,
                     grouping=(P, c, rounds), permissions=RE, flags=flags, input_subnormals=modes[0],
                     result_subnormals=modes[1])
        sfx = FORMS[form] + ("" if modes == (KEEP, KEEP) else "_m")
        assert rz.symbols == [f"tiler_sum_f32_cooperative{sfx}"], modes


def test_a_prologue_is_a_rule():
    """Under the preserving modes too: its combines are the general ones."""
    def symbol(rows, P, c, modes):
        return realize(L.PROGRAM_FOLD, (rows, P * c), rank=2, grouping=(2, P, c), topology=L.SUM_COOPERATIVE,
                       variant=L.FOLD_FMA, scalars=(0x3F800000, 0), permissions=RE, input_subnormals=modes[0],
                       result_subnormals=modes[1]).symbols
    assert symbol(4096, 64, 4, (KEEP, KEEP)) == ["tiler_sum_f32_cooperative_m"]
    assert symbol(4096, 64, 4, (FS, FS)) == ["tiler_sum_f32_cooperative_packed_m"]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,P,c,rounds,major,forms", CASES)
@pytest.mark.parametrize("modes", [(KEEP, KEEP), (FS, FS), (FS, KEEP), (KEEP, FS), (FP, FS), (FS, FP)])
def test_grouped_sums(ctx, rows, P, c, rounds, major, forms, modes):
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
