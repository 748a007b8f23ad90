"""Tall Q8_0 products whose K is not a multiple of the fp16 GEMM's 128-value
step: the operands get zeros up to the next step, unless the call may not
take the staging that needs (no-allocation entry, open capture), when the
packed weight is decoded in the GEMM's loader as before."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROW_REL_L2 = 1e-3     # operands rounded to fp16: the bar of the other tall products
LOADER = b"gemm_f16mfma_128x128x32_q8_0"


def row_rel(a, b):
    return (np.linalg.norm(a - b, axis=1) / np.maximum(np.linalg.norm(b, axis=1), 1e-30)).max()


def operands(oracle, m, n, k, seed):
    rng = np.random.default_rng(seed)
    w = oracle.quantize(oracle.Q8_0, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    return w, rng.standard_normal((m, k)).astype(np.float32)


# K: one block past a step, one short of it, the edges of the staging's
# register forms (1024, 2048, 5120 padded values) and past the last
@pytest.mark.parametrize("m,n,k,stride", [(1300, 200, 416, None), (1153, 259, 992, None), (1153, 131, 1056, 1057),
                                          (1153, 131, 2016, 2048), (1280, 70, 5088, None), (1281, 65, 5088, 5089),
                                          (1281, 65, 5152, None), (1281, 65, 5152, 5153), (257, 1300, 160, 164),
                                          (257, 410, 160, None), (300, 259, 800, 801), (1152, 100, 1056, None)])
def test_padded_k(gpu_ctx, samhip, oracle, m, n, k, stride):
    print("case padded k", m, n, k, stride, flush=True)
    w, x = operands(oracle, m, n, k, m + n + k)
    rows = np.unique(np.linspace(0, m - 1, 67).astype(int))
    y = gpu_ctx.matmul(8, w, x, x_row_stride=stride)
    assert gpu_ctx.query().kernel_variant.startswith(b"gemm_f16pipe")
    assert row_rel(y[rows], oracle.mul_mat_native(oracle.Q8_0, w, np.ascontiguousarray(x[rows]), oracle.ROUND_X86)) <= ROW_REL_L2
    with samhip.Context(0, samhip.COMPUTE_F16) as f16:
        yf = f16.matmul(8, w, x, x_row_stride=stride)
    ref = x[rows].astype(np.float64) @ oracle.dequantize(8, w, k).astype(np.float64).T
    assert row_rel(yf[rows], ref) <= ROW_REL_L2


def test_padded_k_at_scratch_limits(samhip, oracle):
    """Where the padded operands do not fit (64 MB fixed scratch; a capture
    that may not allocate) the product still runs, in the loader's form."""
    print("case padded k at scratch limits", flush=True)
    m, n, k = 6500, 1024, 4704
    w, x = operands(oracle, m, n, k, 3)
    with samhip.Context(0) as ctx:
        wb, xb = ctx.upload(w), ctx.upload(x)
        ya, yb = ctx.alloc(m * n * 4), ctx.alloc(m * n * 4)
        W, X = samhip.tensor(8, k, n, wb.ptr), samhip.tensor(samhip.F32, k, m, xb.ptr)
        Ya, Yb = samhip.tensor(samhip.F32, n, m, ya.ptr), samhip.tensor(samhip.F32, n, m, yb.ptr)
        samhip.check(samhip.lib().samhip_mul_mat_noalloc(ctx.handle, ctypes.byref(W), ctypes.byref(X), ctypes.byref(Yb)))
        assert ctx.query().kernel_variant == LOADER
        ctx.mul_mat(W, X, Ya)
        assert ctx.query().kernel_variant.startswith(b"gemm_f16pipe")
        a, b = ctx.download(ya, (m, n), np.float32), ctx.download(yb, (m, n), np.float32)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))   # the same operands, summed in the same order
    # a context whose staging holds the activations but not the weight too
    m, n, k = 1300, 900, 1056
    w, x = operands(oracle, m, n, k, 4)
    with samhip.Context(0) as ctx:
        ref = ctx.matmul(8, w, x)
    with samhip.Context(0) as ctx:
        wb, xb, yb = ctx.upload(w), ctx.upload(x), ctx.alloc(m * n * 4)
        W, X, Y = samhip.tensor(8, k, n, wb.ptr), samhip.tensor(samhip.F32, k, m, xb.ptr), samhip.tensor(samhip.F32, n, m, yb.ptr)
        # 257 + 20 rows of 5248 padded halves, 2.9 MB, reserve 3 MB
        small_w, small_x = operands(oracle, 257, 20, 5152, 5)
        ctx.matmul(8, small_w, small_x)
        ctx.capture_begin()
        ctx.mul_mat(W, X, Y)
        graph = ctx.capture_end()
        assert ctx.query().kernel_variant == LOADER
        for _ in range(3):
            ctx.write(yb, np.zeros((m, n), np.float32))
            graph.launch()
            ctx.synchronize()
            assert np.array_equal(ctx.download(yb, (m, n), np.float32).view(np.uint32), ref.view(np.uint32))
        graph.destroy()


# SAMHIP_TALL_DECODE=1: a ring of K steps in registers up to a tile per CU
# (256), one step past that; steps of 32 values fewer than the ring holds, and
# left over after whole turns of it
@pytest.mark.parametrize("m,n", [(300, 1031), (2200, 2100)])
@pytest.mark.parametrize("qtype,k", [(8, 64), (8, 96), (8, 160), (8, 288), (12, 256), (13, 512), (14, 256)])
def test_in_loader_decode_has_the_bits_of_the_staged_weight(gpu_ctx, samhip, oracle, monkeypatch, qtype, m, n, k):
    print("case in-loader decode", qtype, m, n, k, flush=True)
    rng = np.random.default_rng(m + n + k)
    w = oracle.quantize(qtype, (rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = gpu_ctx.matmul(qtype, w, x)
    assert gpu_ctx.query().kernel_variant.startswith(b"gemm_f16pipe")
    monkeypatch.setenv("SAMHIP_TALL_DECODE", "1")
    with samhip.Context(0) as ctx:
        z = ctx.matmul(qtype, w, x)
        assert ctx.query().kernel_variant.startswith(b"gemm_f16mfma_128x128x32")
    assert np.array_equal(y.view(np.uint32), z.view(np.uint32))
