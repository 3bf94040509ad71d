"""The value contraction's right operand stored [k, n] (transposed ahead of the
MFMA kernels): 16-byte and 2-byte forms of the transpose at the edges of its
64 x 64 tiles, and its scratch across calls of growing and shrinking size.
Operands are small integers, so the results are exact whatever the order."""
import numpy as np
import pytest

import oracle
from tiler_amd import _lib as L

pytestmark = pytest.mark.gpu


def _check(ctx, m, k, n, batches=3, stream=None):
    rng = np.random.default_rng(m + 3 * k + n)
    p = rng.integers(-3, 4, (batches, m, k)).astype(np.float32)
    v = rng.integers(-3, 4, (batches, k, n)).astype(np.float32)
    want = np.matmul(p.astype(np.float64), v.astype(np.float64)).astype(np.float32)
    s = L.contraction_structure("bmk", p.shape, "bkn", v.shape, "bmn")
    bufs = [ctx.to_device(oracle.bf16_narrow(p)), ctx.to_device(oracle.bf16_narrow(v)), ctx.alloc(want.size * 2)]
    try:
        ctx.contract(L.BF16, s, *bufs, permissions=L.PERMITS_REASSOCIATION, stream=stream)
        ctx.synchronize()
        got = bufs[2].download(np.uint16, want.shape)
    finally:
        for b in bufs:
            b.free()
    assert np.array_equal(got, oracle.bf16_narrow(want).reshape(want.shape))


@pytest.mark.parametrize("k,n", [(64, 64), (72, 40), (8, 8), (136, 128), (200, 72),  # 16 bytes a lane
                                 (65, 64), (64, 41), (7, 3)])                        # 2 bytes
def test_transposed_right_operand(ctx, k, n):
    _check(ctx, 5, k, n)


def test_scratch_across_sizes(ctx):
    for k, n in ((64, 64), (1024, 520), (64, 72), (2048, 1032), (40, 8), (1024, 520)):
        _check(ctx, 9, k, n, batches=2)


def test_scratch_of_other_streams_and_threads(ctx):
    """Calls on another stream take scratch of their own; two threads with a
    context each run at once, and take turns on a shared one (calls on one
    context never overlap)."""
    import threading

    import tiler_amd
    with tiler_amd.Context(0) as other:
        for _ in range(4):
            _check(ctx, 33, 520, 136)  # the context's stream
            rng = np.random.default_rng(5)
            p = rng.integers(-3, 4, (2, 7, 72)).astype(np.float32)
            v = rng.integers(-3, 4, (2, 72, 40)).astype(np.float32)
            want = np.matmul(p, v)
            s = L.contraction_structure("bmk", p.shape, "bkn", v.shape, "bmn")
            bufs = [ctx.to_device(oracle.bf16_narrow(p)), ctx.to_device(oracle.bf16_narrow(v)),
                    ctx.alloc(want.size * 2)]
            ctx.contract(L.BF16, s, *bufs, permissions=L.PERMITS_REASSOCIATION, stream=other.stream)
            other.synchronize()
            got = bufs[2].download(np.uint16, want.shape)
            for b in bufs:
                b.free()
            assert np.array_equal(got, oracle.bf16_narrow(want).reshape(want.shape))
    errors, turn = [], threading.Lock()

    def work(k, n):
        try:
            with tiler_amd.Context(0) as own:
                for _ in range(4):
                    _check(own, 17, k, n)
                    with turn:
                        _check(ctx, 17, k, n)
        except BaseException as e:  # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in ((520, 264), (72, 1032))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_kept_widening_is_exact(ctx):
    """Results of 48 MiB and up take the form with ordinary stores."""
    n = (12 << 20) + 5
    x = np.random.default_rng(3).integers(0, 1 << 16, n).astype(np.uint16)
    dx, dy = ctx.to_device(x), ctx.alloc(4 * n)
    try:
        ctx.convert(L.CONVERT_WIDEN_BF16_F32, dx, n, dy)
        ctx.synchronize()
        got = dy.download(np.uint32, (n,))
    finally:
        dx.free()
        dy.free()
    assert np.array_equal(got, x.astype(np.uint32) << 16)


@pytest.mark.parametrize("n", [(12 << 20) - 4, 12 << 20, (1 << 25) + 3, (1 << 25) + 4])
def test_kept_maps_are_exact(ctx, n):
    """The scaling and adding maps one 16-byte chunk below 48 MiB of result (the
    streaming loop), at 48 and at 128 MiB (ordinary stores; the last with a
    tail), and one chunk past them (streaming again)."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    z = np.ascontiguousarray(x[::-1])
    dx, dz, dy = ctx.to_device(x), ctx.to_device(z), ctx.alloc(4 * n + 16)
    try:
        for call, want in ((lambda: ctx.map(L.MAP_SCALE_BIAS, L.F32, dx, n, dy, a=0.75, b=-2.0),
                            x * np.float32(0.75) + np.float32(-2.0)),
                           (lambda: ctx.map(L.MAP_ADD, L.F32, dx, n, dy, x2=dz), x + z)):
            ctx.fill_u32(dy, 0x7FC12345, n + 4)
            call()
            ctx.synchronize()
            got = dy.download(np.uint32, (n + 4,))
            assert np.array_equal(got[:n], want.view(np.uint32))
            assert (got[n:] == 0x7FC12345).all()
    finally:
        for b in (dx, dz, dy):
            b.free()
