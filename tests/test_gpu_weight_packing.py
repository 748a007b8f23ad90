"""K-quant packing at the edges of its launch: super-block counts that leave a
wave partly idle, sources and destinations off the wide accesses' alignment,
and the blocks whose scale search ends early, byte for byte against the
oracle."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def special_rows(rows, k, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((rows, k)) * 0.02).astype(np.float32)
    blocks = w.reshape(-1, 32)
    forms = [np.zeros(32), np.full(32, 0.25), np.full(32, -0.25), np.full(32, 1e-20), np.linspace(-1e30, 1e30, 32),
             np.abs(blocks[0]), -np.abs(blocks[0]), np.where(np.arange(32) == 17, 5.0, 0.0)]
    # every form among ordinary sub-blocks, and a super-block that holds nothing else of its kind
    for i, f in enumerate(forms):
        blocks[(11 * i + 3) % len(blocks)] = f
    if len(blocks) >= 48:
        blocks[24:32] = 0.0
        blocks[32:40] = 1e-20
        blocks[40:48] *= 1e-12
    return w


@pytest.mark.parametrize("qtype", [12, 13, 14])
@pytest.mark.parametrize("rows,k,src_off,stride_pad,dst_off",
                         [(1, 256, 0, 0, 0), (3, 256, 0, 0, 2), (7, 768, 4, 0, 0), (5, 1280, 0, 1, 1), (257, 512, 0, 4, 4)])
def test_weight_packing_edges(gpu_ctx, oracle, qtype, rows, k, src_off, stride_pad, dst_off):
    print("case weight packing", qtype, rows, k, src_off, stride_pad, dst_off, flush=True)
    w = special_rows(rows, k, 100 * qtype + rows)
    stride = k + stride_pad
    src = np.zeros((rows, stride), np.float32)
    src[:, :k] = w
    sbuf = gpu_ctx.alloc(src.nbytes + 16)
    gpu_ctx.write(sbuf, src, src_off)
    ref = oracle.quantize(qtype, w)
    room = np.full(ref.size + dst_off + 64, 0xA5, np.uint8)
    dbuf = gpu_ctx.upload(room)
    gpu_ctx.quantize_rows(qtype, sbuf.ptr + src_off, 4 * stride, dbuf.ptr + dst_off, rows, k)
    got = gpu_ctx.download(dbuf, room.shape, np.uint8)
    assert np.array_equal(got[dst_off:dst_off + ref.size], ref.reshape(-1))
    assert (got[:dst_off] == 0xA5).all() and (got[dst_off + ref.size:] == 0xA5).all()
    sbuf.free()
    dbuf.free()
