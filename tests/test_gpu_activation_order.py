"""Activation blocks whose packing depends on the order of their elements or
leaves the finite range of its reciprocals: the largest magnitude reached with
both signs (Q8_K keeps the first), blocks of tiny values, NaN and infinite
values beside them.  The staging and every kernel that packs activations
itself, against the oracle's native products."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def activations(m, k, kind):
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if kind == "ties":
        x = np.round(2 * x)              # +-amax in most blocks, in either order
        x[::3] = np.sign(x[::3])
        x[1, :256], x[1, 0], x[1, 255] = 0.25, -3.0, 3.0
        x[2, :256], x[2, 0], x[2, 255] = 0.25, 3.0, -3.0
    elif kind == "tiny":                 # block maxima from 2^-125 to 2^-85
        x = np.clip(x, -4, 4) * 2.0 ** rng.integers(-123, -87, (m, 1))
        x[:, ::5] = 0.0
    return x.astype(np.float32)


def row_rel(y, ref):
    return (np.linalg.norm(y.astype(np.float64) - ref, axis=1) / np.maximum(np.linalg.norm(ref.astype(np.float64), axis=1), 1e-36)).max()


# (m, n, k): staging (one wave a row, two waves a row), int8 strip, fused, small-weight kernel
@pytest.mark.parametrize("m,n,k,bar", [(300, 300, 512, 1e-3), (300, 40, 4608, 1e-3), (32, 96, 1024, 2e-5), (200, 1300, 512, 1e-3),
                                       (300, 100, 256, 2e-5)])
@pytest.mark.parametrize("qtype", [8, 12, 14])
def test_tied_blocks(gpu_ctx, oracle, qtype, m, n, k, bar):
    print("case tied blocks", qtype, m, n, k, flush=True)
    w = oracle.quantize(qtype, (np.random.default_rng(n).standard_normal((n, k)) * 0.02).astype(np.float32))
    x = activations(m, k, "ties")
    y = gpu_ctx.matmul(qtype, w, x)
    assert row_rel(y, oracle.mul_mat_native(qtype, w, x, oracle.ROUND_X86)) <= bar


@pytest.mark.parametrize("m,n,k", [(300, 300, 512), (300, 40, 4608), (200, 1300, 512)])
def test_tiny_and_non_finite_rows(gpu_ctx, oracle, m, n, k):
    """Rows staged as fp16 under their own power of two: tiny K-quant rows as
    the oracle has them (their products stay normal floats), and a NaN or an
    infinity changes no other row."""
    print("case tiny and non-finite rows", m, n, k, flush=True)
    w = oracle.quantize(12, np.random.default_rng(n).standard_normal((n, k)).astype(np.float32))
    x = activations(m, k, "tiny")
    x[: m // 2] *= np.float32(2.0 ** 30)
    x[m // 2:] = activations(m, k, "plain")[m // 2:]
    ref = oracle.mul_mat_native(12, w, x, oracle.ROUND_X86)
    y = gpu_ctx.matmul(12, w, x)
    assert row_rel(y * np.float32(2.0 ** 60), ref * np.float32(2.0 ** 60)) <= 1e-3
    bad = [3, m // 2 + 1, m - 1]
    x2 = x.copy()
    x2[bad[0], 7], x2[bad[1], k - 1], x2[bad[2], 300] = np.nan, np.inf, -np.inf
    y2 = gpu_ctx.matmul(12, w, x2)
    keep = np.setdiff1d(np.arange(m), bad)
    assert np.array_equal(y2[keep].view(np.uint32), y[keep].view(np.uint32))
