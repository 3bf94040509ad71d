"""The strict f32 contraction's column-per-lane forms (1, 4 and 16 rows to 64
columns) and the 64 x 64 tiles, at the edges of their tiles and of the 64-step
stages of k, bit for bit with the oracle's first-product fold
(tiler-reference/src/contraction.rs:558-630)."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L
from tiler_amd.realize import realize

CASES = [
    (17, 63, 64, "b16"), (18, 65, 65, "b16"), (20, 64, 128, "b16"), (33, 130, 191, "b16"), (19, 7, 260, "b16"),
    (10, 2049, 128, "s64"), (16, 1000, 191, "s64"), (2, 8191, 66, "s64"), (9, 1100, 1024, "s64"),
    (250, 1030, 100, "b32"), (273, 1000, 131, "b32"), (289, 2049, 64, "b32"), (2048, 2047, 66, "b64"),
]


@pytest.mark.parametrize("m,n,k,form", CASES)
def test_form_choice(m, n, k, form):
    rz = realize(L.PROGRAM_CONTRACTION, (m, n, k))
    assert rz.symbols == [f"tiler_contract_strict_f32_{form}"]


def test_long_k_keeps_64_bit_addresses():
    assert realize(L.PROGRAM_CONTRACTION, (17, 2, 1 << 24)).symbols == ["tiler_contract_strict_f32_b64"]
    assert realize(L.PROGRAM_CONTRACTION, (16, 1 << 20, 1 << 24)).symbols == ["tiler_contract_strict_f32_s16"]


@pytest.mark.parametrize("m,n,k,form", [
    # many rounds, or ragged k: the 64 x 64 tiles; few rounds: 16 rows a workgroup
    (3000, 4492, 1001, "b64"), (2564, 4492, 161, "b64"), (1500, 4492, 127, "b64"), (3000, 1000, 1001, "b64"),
    (3000, 4492, 64, "b64"), (1024, 3072, 1024, "b32"), (512, 3072, 1024, "b32"), (2102, 203, 65, "b32"),
    (1566, 1800, 448, "b32"),
])
def test_large_products(m, n, k, form):
    assert realize(L.PROGRAM_CONTRACTION, (m, n, k)).symbols == [f"tiler_contract_strict_f32_{form}"]


def test_wide_n_stays_within_the_grid():
    """2^32 work items along n do not fit a launch; a 64 x 64 tile per 256 threads does."""
    assert realize(L.PROGRAM_CONTRACTION, (17, (1 << 28) - 64, 64)).symbols == ["tiler_contract_strict_f32_b32"]
    assert realize(L.PROGRAM_CONTRACTION, (17, 1 << 28, 64)).symbols == ["tiler_contract_strict_f32_b64"]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,form", CASES)
def test_columns_match_the_strict_fold(ctx, m, n, k, form):
    rng = np.random.default_rng(m * 7 + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k)).astype(np.float32)
    a[m - 1] = -0.0                      # products of zeros keep their sign through the seed
    b[0] = np.abs(b[0])
    a[0, k - 1], b[n - 1, 0] = np.inf, np.nan
    a[m // 2] *= np.float32(1e-30)
    b[n // 2] *= np.float32(1e-12)       # subnormal products
    want = oracle.contract_strict_f32(a, b, m, n, k).reshape(m, n)
    dc = ctx.alloc(4 * m * n + 64)
    padded = np.concatenate([np.zeros(1, np.float32), b.reshape(-1)])
    for off in (0, 4):                   # b 16-byte aligned, then 4-byte
        da, db = ctx.to_device(a), ctx.to_device(padded if off else b)
        try:
            ctx.fill_u32(dc, 0x7FC12345, m * n + 16)
            ctx.contract_strict_f32(da, db.offset(off), m, n, k, dc)
            ctx.synchronize()
            got = dc.download(np.uint32, (m * n + 16,))
        finally:
            da.free()
            db.free()
        assert np.array_equal(got[:m * n], want.view(np.uint32).reshape(-1)), (form, off)
        assert (got[m * n:] == 0x7FC12345).all()
    dc.free()
