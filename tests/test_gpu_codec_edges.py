"""Row decoding and Q8_0 packing at the edges of their launches: rows shorter
than a workgroup's run, widths that leave part of one, more rows than the
grid holds at once, and sources and destinations off the wide accesses'
alignment; bit for bit against the oracle."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(rows, k, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((rows, k)) * np.exp(rng.uniform(-6, 6, (rows, 1)))).astype(np.float32)


SHAPES = {8: [(1, 32), (67, 96), (3, 1056), (5, 4736), (33000, 32)], 12: [(1, 256), (9, 1280), (3, 4608)],
          13: [(7, 768)], 14: [(1, 256), (9, 1280)], 15: [(5, 1280)], 1: [(1, 32), (67, 96), (3, 1056)]}


@pytest.mark.parametrize("qtype,rows,k", [(t, r, k) for t, shapes in SHAPES.items() for r, k in shapes])
@pytest.mark.parametrize("pad,off", [(0, 0), (2, 2)])
@pytest.mark.parametrize("dst_off", [0, 4])
def test_dequantize_edges(gpu_ctx, oracle, qtype, rows, k, pad, off, dst_off):
    print("case dequantize", qtype, rows, k, pad, off, dst_off, flush=True)
    x = rows_of(rows, k, qtype + rows)
    if qtype == 1:
        packed, ref = x.astype(np.float16).view(np.uint8).reshape(rows, -1), x.astype(np.float16).astype(np.float32)
    else:
        packed = oracle.quantize(qtype, x, oracle.ROUND_REF).reshape(rows, -1)
        ref = oracle.dequantize(qtype, packed, k)
    rb = packed.shape[1]
    src = np.zeros((rows, rb + pad), np.uint8)
    src[:, :rb] = packed
    sbuf = gpu_ctx.alloc(src.nbytes + 16)
    gpu_ctx.write(sbuf, src, off)
    room = np.full(ref.size + 8, 7.0, np.float32)
    dbuf = gpu_ctx.upload(room)
    gpu_ctx.dequantize_rows(qtype, sbuf.ptr + off, rb + pad, dbuf.ptr + dst_off, rows, k)
    got = gpu_ctx.download(dbuf, room.shape, np.float32)
    at = dst_off // 4
    assert np.array_equal(got[at:at + ref.size].view(np.uint32), ref.reshape(-1).view(np.uint32))
    assert (got[:at] == 7.0).all() and (got[at + ref.size:] == 7.0).all()
    sbuf.free()
    dbuf.free()


@pytest.mark.parametrize("rounding", ["x86", "ref"])
@pytest.mark.parametrize("rows,k,src_off,pad,dst_off", [(1, 32, 0, 0, 0), (5, 96, 0, 0, 2), (7, 1056, 4, 0, 0),
                                                        (9, 544, 0, 1, 1), (3, 4736, 0, 4, 4)])
def test_quantize_q8_0_edges(gpu_ctx, oracle, samhip, rounding, rows, k, src_off, pad, dst_off):
    print("case quantize q8_0", rounding, rows, k, src_off, pad, dst_off, flush=True)
    x = rows_of(rows, k, rows + k)
    x[0, :32] = 0.0
    # a tiny block; 127 / amax stays finite down to amax = 127 / FLT_MAX = 3.8e-37, and below that the
    # packers convert an infinity to int, which C leaves undefined
    x[-1, -32:] = 1e-36
    src = np.zeros((rows, k + pad), np.float32)
    src[:, :k] = x
    sbuf = gpu_ctx.alloc(src.nbytes + 16)
    gpu_ctx.write(sbuf, src, src_off)
    ref = oracle.quantize(8, x, oracle.ROUND_X86 if rounding == "x86" else oracle.ROUND_REF).reshape(-1)
    room = np.full(ref.size + dst_off + 64, 0xA5, np.uint8)
    dbuf = gpu_ctx.upload(room)
    gpu_ctx.quantize_rows(8, sbuf.ptr + src_off, 4 * (k + pad), dbuf.ptr + dst_off, rows, k,
                          samhip.ROUND_X86 if rounding == "x86" else samhip.ROUND_REF)
    got = gpu_ctx.download(dbuf, room.shape, np.uint8)
    assert np.array_equal(got[dst_off:dst_off + ref.size], ref)
    assert (got[:dst_off] == 0xA5).all() and (got[dst_off + ref.size:] == 0xA5).all()
    sbuf.free()
    dbuf.free()


@pytest.mark.parametrize("rounding", ["x86", "ref"])
def test_quantize_q8_0_nan_blocks(gpu_ctx, samhip, rounding):
    """NaN packs as code 0; a block of nothing else keeps a NaN scale, one with a finite value that value's."""
    x = np.full((3, 64), np.nan, np.float32)
    x[1, 5] = -127.0
    x[2] = 1.0
    got = gpu_ctx.quantize(8, x, samhip.ROUND_X86 if rounding == "x86" else samhip.ROUND_REF).reshape(3, 2, 34)
    scale = np.ascontiguousarray(got[:, :, :2]).view(np.float16)[:, :, 0]
    assert np.isnan(scale[0]).all() and scale[1, 0] == 1.0 and np.isnan(scale[1, 1])
    codes = got[:, :, 2:].view(np.int8)
    assert (codes[0] == 0).all() and codes[1, 0, 5] == -127 and np.count_nonzero(codes[1]) == 1 and (codes[2] == 127).all()
