"""The k-split contraction tiles: every tile at the edges of its blocks (rows
past m, columns past n, n off the 8-element grid, k ragged against the 64-deep
chunks and the waves), bit for bit.  Operands are small integers, so every
product and every partial sum is exact in binary32 whatever the order, and the
output is the exact sum narrowed once."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L
from tiler_amd.realize import realize

RE = L.PERMITS_REASSOCIATION

# (m, n, k, the tile the planner takes for it on 256 CUs)
CASES = [
    (1, 16, 8, "skinny1"), (16, 17, 520, "skinny1"), (7, 130, 72, "skinny1"), (31, 100, 1000, "skinny2"),
    (33, 24, 512, "skinny3"), (64, 1001, 584, "skinny4"), (49, 136, 64, "skinny4"),
    (65, 64, 512, "k2x2"), (97, 121, 1032, "k2x2"), (129, 2001, 520, "k2x4"), (66, 4100, 584, "k2x4"),
    (100, 4104, 520, "k3x4"), (500, 1999, 1000, "k4x4"), (201, 4100, 520, "k5x4"), (1300, 1001, 512, "k6x4"),
    (1000, 1999, 1000, "k4x8"), (490, 4100, 1032, "k6x8"),
]


@pytest.mark.parametrize("m,n,k,form", CASES)
def test_tile_choice(m, n, k, form):
    for variant, silu in ((L.EPILOGUE_NONE, ""), (L.EPILOGUE_SILU, "silu_")):
        rz = realize(L.PROGRAM_CONTRACTION, (m, n, k), dtype=L.BF16, permissions=RE, variant=variant)
        assert rz.symbols == [f"tiler_contract_bf16_{silu}{form}"]


def test_long_k_keeps_the_skinny_form():
    """From k = 2^24 on, 128 rows leave a buffer's 32-bit offsets: the skinny
    forms with 64-bit addresses, for the library's choice and on request."""
    def symbol(m, k, **kw):
        return realize(L.PROGRAM_CONTRACTION, (m, 40, k), dtype=L.BF16, permissions=RE, **kw).symbols
    for form in (L.FORM_AUTO, L.FORM_CONTRACT_SKINNY):
        assert symbol(33, (1 << 24) - 8, form=form) == ["tiler_contract_bf16_skinny3"]
        assert symbol(33, 1 << 24, form=form) == ["tiler_contract_bf16_skinny3_l"]
    assert symbol(64, 1 << 24, variant=L.EPILOGUE_SILU) == ["tiler_contract_bf16_silu_skinny4_l"]
    assert symbol(65, 1 << 24) == ["tiler_contract_bf16_g128"]
    s = L.contraction_structure("bmk", (2, 16, 1 << 24), "nk", (40, 1 << 24), "bmn")
    assert realize(L.PROGRAM_CONTRACTION, (), dtype=L.BF16, structure=s, permissions=RE).symbols == \
        ["tiler_contract_bf16_skinny1_l_b"]
    # 2^32 work items do not fit a launch: the 128-tiles
    assert realize(L.PROGRAM_CONTRACTION, (1, (1 << 27) - 256, 8), dtype=L.BF16, permissions=RE).symbols == \
        ["tiler_contract_bf16_skinny1"]
    assert not realize(L.PROGRAM_CONTRACTION, (1, 1 << 27, 8), dtype=L.BF16,
                       permissions=RE).symbols[0].startswith("tiler_contract_bf16_skinny")


def test_staged_tiles_keep_the_large_products():
    # the last three: several rounds of 128-tiles, and panels that leave some XCDs a second round
    for shape in ((4096, 4096, 4096), (2048, 4096, 4096), (1000, 2048, 512), (3000, 8192, 1024),
                  (3000, 4096, 4096), (1536, 3000, 3400), (1045, 2536, 2248)):
        rz = realize(L.PROGRAM_CONTRACTION, shape, dtype=L.BF16, permissions=RE)
        assert rz.symbols[0].startswith(("tiler_contract_bf16_t256", "tiler_contract_bf16_t128")), shape
    # n off the 8-element grid: the general tiles
    for shape in ((3000, 2049, 1024), (3000, 1001, 512), (4000, 513, 512), (2178, 1278, 1840)):
        rz = realize(L.PROGRAM_CONTRACTION, shape, dtype=L.BF16, permissions=RE)
        assert rz.symbols == ["tiler_contract_bf16_g128"], shape


def _operands(rng, m, n, k):
    a = rng.integers(-3, 4, (m, k)).astype(np.float32)
    b = rng.integers(-3, 4, (n, k)).astype(np.float32)
    return a, b, (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,form", CASES)
@pytest.mark.parametrize("silu", [False, True])
def test_tiles_are_exact_on_integers(ctx, m, n, k, form, silu):
    rng = np.random.default_rng(m * 31 + n + k)
    a, b, want = _operands(rng, m, n, k)
    if silu:
        want = oracle.silu_f32(want.reshape(-1)).reshape(m, n)
    da, db = ctx.to_device(oracle.bf16_narrow(a)), ctx.to_device(oracle.bf16_narrow(b))
    dc = ctx.alloc(m * n * 2 + 68)
    try:
        for off in (0, 2):  # the output 16-byte aligned, then 2-byte
            ctx.fill_u32(dc, 0x7FC17FC1, (m * n * 2 + 68) // 4)
            ctx.contract_bf16(da, db, m, n, k, dc.offset(off), L.EPILOGUE_SILU if silu else L.EPILOGUE_NONE)
            ctx.synchronize()
            raw = dc.download(np.uint16, (m * n + 32,))
            at = off // 2
            assert np.array_equal(raw[at:at + m * n].reshape(m, n), oracle.bf16_narrow(want).reshape(m, n))
            assert (raw[:at] == 0x7FC1).all() and (raw[at + m * n:] == 0x7FC1).all()
    finally:
        da.free()
        db.free()
        dc.free()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(5, 40, 72), (40, 256, 1032), (130, 72, 520), (200, 1000, 584)])
def test_batched_tiles_are_exact_on_integers(ctx, m, n, k):
    """Three problems of A over one shared B ([b, m, k] x [n, k]), fewer and
    more than eight panels of B."""
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-3, 4, (3, m, k)).astype(np.float32)
    b = rng.integers(-3, 4, (n, k)).astype(np.float32)
    want = np.einsum("bmk,nk->bmn", a.astype(np.float64), b.astype(np.float64)).astype(np.float32)
    s = L.contraction_structure("bmk", a.shape, "nk", b.shape, "bmn")
    rz = realize(L.PROGRAM_CONTRACTION, (), dtype=L.BF16, structure=s, permissions=RE)
    assert rz.symbols[0].endswith("_b") and ("skinny" in rz.symbols[0] or "bf16_k" in rz.symbols[0]), rz.symbols
    bufs = [ctx.to_device(oracle.bf16_narrow(a)), ctx.to_device(oracle.bf16_narrow(b)), ctx.alloc(want.size * 2)]
    try:
        ctx.contract(L.BF16, s, *bufs, permissions=RE)
        ctx.synchronize()
        got = bufs[2].download(np.uint16, want.shape)
    finally:
        for x in bufs:
            x.free()
    assert np.array_equal(got, oracle.bf16_narrow(want).reshape(want.shape))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(6, 20, (1 << 24) + 8), (20, 7, 1 << 24), (40, 17, (1 << 24) + 72),
                                   (50, 3, (1 << 24) + 56)])
def test_long_k_is_exact_on_integers(ctx, m, n, k):
    """Operands are nonzero in one element of 4096, so every partial sum stays
    a binary32 integer; among them the last elements of the last row, which lie
    past 2^32 bytes of k from the first one's in the larger cases."""
    rng = np.random.default_rng(m + n)
    at = np.unique(np.concatenate([rng.integers(0, k, k // 4096), np.arange(k - 9, k), np.arange(9)]))
    av = rng.integers(-3, 4, (m, at.size)).astype(np.float32)
    bv = rng.integers(-3, 4, (n, at.size)).astype(np.float32)
    want = (av.astype(np.float64) @ bv.astype(np.float64).T).astype(np.float32)
    a, b = np.zeros((m, k), np.uint16), np.zeros((n, k), np.uint16)
    a[:, at], b[:, at] = oracle.bf16_narrow(av).reshape(av.shape), oracle.bf16_narrow(bv).reshape(bv.shape)
    s = L.contraction_structure("bmk", (2, m // 2, k), "nk", (n, k), "bmn")
    da, db, dc = ctx.to_device(a), ctx.to_device(b), ctx.alloc(m * n * 2)
    try:
        for call in (lambda: ctx.contract_bf16(da, db, m, n, k, dc),
                     lambda: ctx.contract(L.BF16, s, da, db, dc, permissions=RE)):
            ctx.fill_u32(dc, 0x7FC17FC1, m * n * 2 // 4)
            call()
            ctx.synchronize()
            assert np.array_equal(dc.download(np.uint16, (m, n)), oracle.bf16_narrow(want).reshape(m, n))
    finally:
        da.free()
        db.free()
        dc.free()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(20, 40, 520), (130, 120, 584)])
def test_not_finite_operands(ctx, m, n, k):
    """NaN and infinities reach only their own rows and columns; every NaN
    output is the canonical 0x7fc0.  The last row and column hold the values
    that rows and columns past the end would repeat."""
    rng = np.random.default_rng(k)
    a, b, want = _operands(rng, m, n, k)
    a[m - 1, k - 1], a[3, 0], b[n - 1, k - 1] = np.nan, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32)
    da, db, dc = ctx.to_device(oracle.bf16_narrow(a)), ctx.to_device(oracle.bf16_narrow(b)), ctx.alloc(m * n * 2)
    try:
        ctx.contract_bf16(da, db, m, n, k, dc)
        ctx.synchronize()
        got = dc.download(np.uint16, (m, n))
    finally:
        da.free()
        db.free()
        dc.free()
    assert np.array_equal(got, oracle.bf16_narrow(want).reshape(m, n))
