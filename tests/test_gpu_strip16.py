"""Q4_K / Q5_K products with packed activations and whole K per workgroup:
edges of the 16-row tiles in M and N, every length of a wave's run of steps
(K = 512 .. 1024, .. 2048, past it) with waves left over, unaligned
activations, strided output; against the oracle's native products.  Exact
integer dots and F32 sums in another order than the oracle's."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EXACT = 2e-5
VARIANT = {12: b"skinny_i8mfma16_q4_k", 13: b"skinny_i8mfma16_q5_k"}


def row_rel(y, ref):
    return (np.linalg.norm(y.astype(np.float64) - ref, axis=1) / np.maximum(np.linalg.norm(ref.astype(np.float64), axis=1), 1e-30)).max()


# (each has at least 128 workgroups of 16 x 16 rows, or 64 up to K = 1024, and is past one launch of the strip kernel)
SHAPES = [(100, 2100, 512, None), (15, 1030, 768, 769), (16, 1024, 1024, None), (17, 1030, 1280, None), (33, 700, 2048, 2052),
          (49, 517, 2304, None), (255, 130, 4096, None), (100, 4733, 1024, None), (31, 4096, 4608, None), (1, 2064, 2048, None)]


@pytest.mark.parametrize("qtype", [12, 13])
@pytest.mark.parametrize("m,n,k,stride", SHAPES)
def test_strip16(samhip, oracle, qtype, m, n, k, stride):
    print("case strip16", qtype, m, n, k, stride, flush=True)
    rng = np.random.default_rng(m + n + k)
    w = oracle.quantize(qtype, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = (rng.standard_normal((m, k)) * np.exp(rng.uniform(-4, 4, (m, 1)))).astype(np.float32)
    x[0, 3] = np.nan                # packs as code 0
    with samhip.Context(0) as ctx:
        y = ctx.matmul(qtype, w, x, x_row_stride=stride)
        assert ctx.query().kernel_variant == VARIANT[qtype]
        ctx.trace_begin()
        again = ctx.matmul(qtype, w, x)
        assert [r[0] for r in ctx.trace_end()] == ["stage_strip_q8_k", VARIANT[qtype].decode()]
    ref = oracle.mul_mat_native(qtype, w, x)
    assert np.isfinite(ref).all() and np.isfinite(y).all() and row_rel(y, ref) <= EXACT
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))


def test_strip16_rows_off_alignment_and_guarded_output(samhip, oracle):
    """Weight rows at a 2-byte aligned address keep the kernels they had, with
    the same values; no byte beside the output rows changes."""
    print("case strip16 alignment", flush=True)
    m, n, k, ldy = 40, 600, 1024, 611
    rng = np.random.default_rng(9)
    w = oracle.quantize(12, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    ref = oracle.mul_mat_native(12, w, x)
    rb = w.shape[1]
    with samhip.Context(0) as ctx:
        for off in (0, 2):
            raw = np.zeros(n * rb + 16, np.uint8)
            raw[off:off + n * rb] = w.reshape(-1)
            wb, xb = ctx.upload(raw), ctx.upload(x)
            room = np.full((m + 1, ldy), 3.0, np.float32)
            yb = ctx.upload(room)
            ctx.mul_mat(samhip.tensor(12, k, n, wb.ptr + off, nb1=rb), samhip.tensor(samhip.F32, k, m, xb.ptr),
                        samhip.tensor(samhip.F32, n, m, yb.ptr, nb1=4 * ldy))
            assert (ctx.query().kernel_variant == VARIANT[12]) == (off == 0)
            got = ctx.download(yb, room.shape, np.float32)
            assert row_rel(got[:m, :n], ref) <= (EXACT if off == 0 else 1e-3)
            assert (got[:m, n:] == 3.0).all() and (got[m] == 3.0).all()
            for b in (wb, xb, yb):
                b.free()


def test_strip16_capture_and_noalloc(samhip, oracle):
    """Replays and the no-allocation entry give the eager call's bits; a
    capture whose staging cannot hold the packed rows is as before."""
    print("case strip16 capture", flush=True)
    m, n, k = 77, 1000, 2048
    rng = np.random.default_rng(10)
    w = oracle.quantize(13, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    with samhip.Context(0) as ctx:
        wb, xb, yb, zb = ctx.upload(w), ctx.upload(x), ctx.alloc(m * n * 4), ctx.alloc(m * n * 4)
        W, X = samhip.tensor(13, k, n, wb.ptr), samhip.tensor(samhip.F32, k, m, xb.ptr)
        Y, Z = samhip.tensor(samhip.F32, n, m, yb.ptr), samhip.tensor(samhip.F32, n, m, zb.ptr)
        ctx.mul_mat(W, X, Y)
        assert ctx.query().kernel_variant == VARIANT[13]
        eager = ctx.download(yb, (m, n), np.float32)
        samhip.check(samhip.lib().samhip_mul_mat_noalloc(ctx.handle, ctypes.byref(W), ctypes.byref(X), ctypes.byref(Z)))
        assert np.array_equal(ctx.download(zb, (m, n), np.float32).view(np.uint32), eager.view(np.uint32))
        ctx.capture_begin()
        ctx.mul_mat(W, X, Y)
        graph = ctx.capture_end()
        for _ in range(3):
            ctx.write(yb, np.zeros((m, n), np.float32))
            ctx.mul_mat(W, X, Z)          # eager work between replays
            ctx.synchronize()
            graph.launch()
            ctx.synchronize()
            assert np.array_equal(ctx.download(yb, (m, n), np.float32).view(np.uint32), eager.view(np.uint32))
        graph.destroy()
    with samhip.Context(0) as ctx:        # nothing reserved: refused or run, as the kernels before it
        wb, xb, yb = ctx.upload(w), ctx.upload(x), ctx.alloc(m * n * 4)
        ctx.capture_begin()
        with pytest.raises(samhip.InvalidArgument, match="staging"):
            ctx.mul_mat(samhip.tensor(13, k, n, wb.ptr), samhip.tensor(samhip.F32, k, m, xb.ptr),
                        samhip.tensor(samhip.F32, n, m, yb.ptr))
        ctx.capture_end().destroy()


@pytest.mark.parametrize("m,n,k", [(255, 130, 4096), (255, 512, 32768)])
def test_strip16_arithmetic_does_not_depend_on_earlier_calls(samhip, oracle, m, n, k):
    """A capture in a context that has only run other products and the
    no-allocation entry give the eager call's bits: those products leave less
    staging than the packed rows take (1.2 and 9.5 MB), but enough for the
    kernels that would otherwise stand in, the exact one with another order
    of sums and the one that rounds its operands to fp16."""
    print("case strip16 history", m, n, k, flush=True)
    rng = np.random.default_rng(n + k)
    w = oracle.quantize(12, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    rows = [0, 1, m // 2, m - 1]
    ref = oracle.mul_mat_native(12, w, np.ascontiguousarray(x[rows]))
    with samhip.Context(0) as ctx:
        eager = ctx.matmul(12, w, x)
    assert row_rel(eager[rows], ref) <= EXACT
    with samhip.Context(0) as ctx:
        if k > 4096:   # 5 MB
            ctx.matmul(8, oracle.quantize(8, np.ones((512, 1024), np.float32)), np.ones((2000, 1024), np.float32))
        else:          # 1 MB
            ctx.matmul(12, w[:64, :144], np.ascontiguousarray(x[:4, :256]))
        assert ctx.query().activation_allocation_peak_bytes < 256 * k * 9 // 8
        wb, xb, yb = ctx.upload(w), ctx.upload(x), ctx.alloc(m * n * 4)
        W, X, Y = samhip.tensor(12, k, n, wb.ptr), samhip.tensor(samhip.F32, k, m, xb.ptr), samhip.tensor(samhip.F32, n, m, yb.ptr)
        ctx.capture_begin()
        ctx.mul_mat(W, X, Y)
        graph = ctx.capture_end()
        for _ in range(2):
            ctx.write(yb, np.zeros((m, n), np.float32))
            graph.launch()
            ctx.synchronize()
            assert np.array_equal(ctx.download(yb, (m, n), np.float32).view(np.uint32), eager.view(np.uint32))
        graph.destroy()
        ctx.write(yb, np.zeros((m, n), np.float32))
        samhip.check(samhip.lib().samhip_mul_mat_noalloc(ctx.handle, ctypes.byref(W), ctypes.byref(X), ctypes.byref(Y)))
        assert np.array_equal(ctx.download(yb, (m, n), np.float32).view(np.uint32), eager.view(np.uint32))


@pytest.mark.parametrize("name,value", [("SAMHIP_INT8_STRIP", "2"), ("SAMHIP_I8_STRIP_ROWS", "32"),
                                        ("SAMHIP_STRIP_SKINNY", "2")])
def test_settings_for_the_strip_kernel_reach_it(samhip, oracle, monkeypatch, name, value):
    """The settings that ask for the one-launch strip kernels give the bits of
    the one that takes this size (its order of sums differs), not those of
    the kernel that is the default."""
    print("case strip settings", name, value, flush=True)
    m, n, k = 32, 1024, 4096
    rng = np.random.default_rng(12)
    w = oracle.quantize(12, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)

    def run(variant):
        with samhip.Context(0) as ctx:
            y = ctx.matmul(12, w, x)
            assert ctx.query().kernel_variant == variant
            return y.view(np.uint32)

    default = run(VARIANT[12])
    monkeypatch.setenv("SAMHIP_STRIP16", "0")
    strip = run(b"skinny_i8mfma_q4_k")
    assert not np.array_equal(default, strip)   # else the last line says nothing
    monkeypatch.delenv("SAMHIP_STRIP16")
    monkeypatch.setenv(name, value)
    assert np.array_equal(run(b"skinny_i8mfma_q4_k"), strip)


@pytest.mark.parametrize("qtype,m,n,k,taken", [(12, 128, 256, 4096, False), (12, 144, 256, 4096, True),
                                               (12, 64, 512, 4096, True), (13, 64, 512, 4096, False),
                                               (13, 32, 1024, 4096, False), (12, 32, 1024, 4096, True),
                                               (13, 16, 2048, 4096, True), (13, 32, 1024, 4608, True),
                                               (13, 64, 4096, 1024, True), (13, 65, 2048, 1024, False),
                                               (12, 33, 4096, 1024, True), (13, 16, 4736, 1024, True)])
def test_strip16_where_it_is_faster(samhip, oracle, qtype, m, n, k, taken):
    """Both sides of the lines of strip16_preferred at half the chip and at K
    in one launch; exact either way."""
    print("case strip16 line", qtype, m, n, k, flush=True)
    rng = np.random.default_rng(m + n + k)
    w = oracle.quantize(qtype, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    with samhip.Context(0) as ctx:
        y = ctx.matmul(qtype, w, x)
        assert ctx.query().kernel_variant == (VARIANT[qtype] if taken else VARIANT[qtype].replace(b"16", b""))
    assert row_rel(y, oracle.mul_mat_native(qtype, w, x)) <= EXACT
