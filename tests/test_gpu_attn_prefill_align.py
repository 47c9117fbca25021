"""attn_prefill_f16 refuses a head stride that leaves K/V rows unaligned (its
copies into LDS are 16 bytes wide), where that stride is used at all."""
import numpy as np
import pytest

from test_gpu_kernels import _assert_attn_close, _dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,rows,off,refused", [(4, 2, 9, 4, True), (4, 2, 9, 1, True), (4, 2, 9, 8, False),
                                                    (4, 1, 9, 1, False), (4, 2, 0, 1, False)])
def test_head_stride_alignment(rf, orc, stream, nh, nkv, rows, off, refused):
    hd, cap = 64, 16
    rng = np.random.default_rng(off)
    hs = cap * hd + off
    q = rng.standard_normal((max(rows, 1), nh * hd)).astype(np.float32)
    kc, vc = (rng.standard_normal(nkv * hs).astype(np.float16).view(np.uint16) for _ in range(2))
    out = rf.DeviceBuffer.zeroed(q.size, np.float32, stream)
    args = (nh, nkv, hd, 0, rows, _dev(rf, q.reshape(-1), stream), nh * hd, _dev(rf, kc, stream), _dev(rf, vc, stream), hd, hs,
            out, nh * hd)
    if refused:
        with pytest.raises(rf.Rfp4Error) as e:
            rf.attn_prefill_f16(stream, *args)
        assert e.value.code == -6
        return
    rf.attn_prefill_f16(stream, *args)
    got = out.to_host(q.size, np.float32, stream).reshape(q.shape)
    if rows:
        _assert_attn_close(got, np.stack([orc.attn_decode(nh, nkv, hd, r + 1, q[r], kc, vc, hd, hs) for r in range(rows)]))
