"""attn_prefill_f16: four key groups of 4 waves and two of 8 (forced and as
planned), scores whose running maximum is raised in most blocks, token-major
caches, and strides past the 32-bit copy offsets, against the oracle's
attn_decode row by row (the bar of test_attn_prefill_f16)."""
import numpy as np
import pytest

from test_gpu_kernels import _assert_attn_close, _dev

pytestmark = pytest.mark.gpu


def _run(rf, orc, stream, nh, nkv, hd, pos0, rows, ksplit=0, token_major=False):
    rng = np.random.default_rng(pos0 * 31 + rows + hd + nh)
    cap = pos0 + rows
    q = rng.standard_normal((rows, nh * hd)).astype(np.float32)
    kc, vc = (rng.standard_normal(nkv * cap * hd).astype(np.float16).view(np.uint16) for _ in range(2))
    ts, hs = (nkv * hd, hd) if token_major else (hd, cap * hd)
    oref = np.stack([orc.attn_decode(nh, nkv, hd, pos0 + r + 1, q[r], kc, vc, ts, hs) for r in range(rows)])
    dout = rf.DeviceBuffer.zeroed(rows * nh * hd, np.float32, stream)
    rf.check(rf.load().rfp4_debug_prefill_ksplit(ksplit))
    try:
        rf.attn_prefill_f16(stream, nh, nkv, hd, pos0, rows, _dev(rf, q.reshape(-1), stream), nh * hd,
                            _dev(rf, kc, stream), _dev(rf, vc, stream), ts, hs, dout, nh * hd)
    finally:
        rf.check(rf.load().rfp4_debug_prefill_ksplit(0))
    _assert_attn_close(dout.to_host(rows * nh * hd, np.float32, stream).reshape(rows, nh * hd), oref)


# fewer blocks than groups, one block each, whole and partial last blocks; 3 heads of a padded group of 4
@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 128), (2, 1, 64), (3, 3, 128), (6, 2, 64), (8, 1, 128), (16, 2, 64)])
@pytest.mark.parametrize("pos0,rows", [(0, 1), (0, 33), (95, 33), (250, 70)])
def test_key_groups(rf, orc, stream, nh, nkv, hd, pos0, rows):
    _run(rf, orc, stream, nh, nkv, hd, pos0, rows, ksplit=2 if nh // nkv == 8 else 4)


# the planner's own choice on both sides of its lines (64, 128, 512 and 1024 keys)
@pytest.mark.parametrize("nh,nkv,hd,pos0,rows", [(4, 1, 64, 0, 64), (4, 1, 64, 0, 65), (4, 1, 64, 0, 128), (2, 1, 64, 100, 29),
                                                 (4, 1, 128, 0, 64), (4, 1, 128, 50, 15), (8, 1, 64, 500, 12), (8, 1, 128, 500, 13),
                                                 (4, 1, 128, 1000, 24), (4, 1, 128, 1000, 25)])
def test_planned_key_groups(rf, orc, stream, nh, nkv, hd, pos0, rows):
    _run(rf, orc, stream, nh, nkv, hd, pos0, rows, token_major=True)


# Scores tens apart: most blocks raise some row's maximum by more than 8.  The
# bound, against float64: a score is a sum of hd products whose q holds a
# relative 2^-22 (hi + lo) and whose f32 sum holds about as much, so it is off
# by at most 2^-21 A, A = sum |q k| / sqrt(hd); a probability is off by that
# factor, and the row by twice it times max |v| (numerator and denominator).
@pytest.mark.parametrize("ksplit", [1, 2, 4])
@pytest.mark.parametrize("hd", [64, 128])
def test_growing_maximum(rf, stream, hd, ksplit):
    nh, pos0, rows = 4, 40, 150
    rng = np.random.default_rng(hd + ksplit)
    cap = pos0 + rows
    q = (12.0 * rng.standard_normal((rows, nh, hd))).astype(np.float32)
    k, v = (rng.standard_normal((cap, hd)).astype(np.float16) for _ in range(2))
    dout = rf.DeviceBuffer.zeroed(rows * nh * hd, np.float32, stream)
    rf.check(rf.load().rfp4_debug_prefill_ksplit(ksplit))
    try:
        rf.attn_prefill_f16(stream, nh, 1, hd, pos0, rows, _dev(rf, q.reshape(-1), stream), nh * hd,
                            _dev(rf, k.view(np.uint16).reshape(-1), stream), _dev(rf, v.view(np.uint16).reshape(-1), stream),
                            hd, cap * hd, dout, nh * hd)
    finally:
        rf.check(rf.load().rfp4_debug_prefill_ksplit(0))
    got = dout.to_host(rows * nh * hd, np.float32, stream).reshape(rows, nh, hd)
    q, k, v = q.astype(np.float64), k.astype(np.float64), v.astype(np.float64)
    s = np.einsum("rhd,td->rht", q, k) / np.sqrt(hd)
    amp = (np.einsum("rhd,td->rht", abs(q), abs(k)) / np.sqrt(hd)).max(-1, keepdims=True)
    s[np.arange(cap)[None, None] > pos0 + np.arange(rows)[:, None, None] + 0 * s] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v
    assert np.all(abs(got - ref) <= 2.0 ** -20 * amp * abs(v).max())


def test_long_token_stride(rf, orc, stream):
    """2^24 halves between tokens: past the copies' 32-bit lane offsets."""
    nh, nkv, hd, rows, ts = 4, 1, 64, 20, 1 << 24
    rng = np.random.default_rng(5)
    q = rng.standard_normal((rows, nh * hd)).astype(np.float32)
    kv = [rng.standard_normal((rows, hd)).astype(np.float16).view(np.uint16) for _ in range(2)]
    bufs = []
    for a in kv:
        b = rf.DeviceBuffer(((rows - 1) * ts + hd) * 2, np.uint16)
        for t in range(rows):
            rf.check(rf.load().rfp4_h2d(b.ptr + 2 * t * ts, a[t].ctypes.data, 2 * hd, stream.h))
        stream.synchronize()
        bufs.append(b)
    oref = np.stack([orc.attn_decode(nh, nkv, hd, r + 1, q[r], kv[0].reshape(-1), kv[1].reshape(-1), hd, rows * hd)
                     for r in range(rows)])
    dout = rf.DeviceBuffer.zeroed(rows * nh * hd, np.float32, stream)
    rf.attn_prefill_f16(stream, nh, nkv, hd, 0, rows, _dev(rf, q.reshape(-1), stream), nh * hd, *bufs, ts, hd, dout, nh * hd)
    _assert_attn_close(dout.to_host(rows * nh * hd, np.float32, stream).reshape(rows, nh * hd), oref)
