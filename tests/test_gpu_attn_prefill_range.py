"""attn_prefill_f16 where the scores are far larger than a softmax needs (finite
q and K of tens of thousands), with rows whose first key block in a key group
is wholly masked: the row of V with the largest score, nothing infinite or NaN."""
import numpy as np
import pytest

from test_gpu_kernels import _dev

pytestmark = pytest.mark.gpu


# The reference is float64.  A score is off by at most 2^-20 A, A = sum |q k| /
# sqrt(hd) (q as two fp16 terms, f32 sums).  The two largest scores of every
# row are more than 2^-18 A apart (asserted), and 2^-19 A is 77 or more here:
# every other probability is below exp(-70), and the output is the V row, exact
# in f32.
@pytest.mark.parametrize("mag", [3000.0, 20000.0])
@pytest.mark.parametrize("nh,nkv,hd,ksplit", [(4, 1, 128, 1), (4, 1, 128, 4), (2, 1, 64, 2), (8, 1, 64, 1), (8, 1, 128, 2)])
def test_large_finite_scores(rf, stream, nh, nkv, hd, ksplit, mag):
    pos0, rows = 40, 90
    cap = pos0 + rows
    rng = np.random.default_rng(int(mag) + hd + nh)
    q = (mag * rng.uniform(-1.5, 1.5, (rows, nh, hd))).astype(np.float32)
    k = (mag * rng.uniform(-1.5, 1.5, (cap, hd))).astype(np.float16)
    v = rng.standard_normal((cap, hd)).astype(np.float16)
    dout = rf.DeviceBuffer.zeroed(rows * nh * hd, np.float32, stream)
    rf.check(rf.load().rfp4_debug_prefill_ksplit(ksplit))
    try:
        rf.attn_prefill_f16(stream, nh, nkv, hd, pos0, rows, _dev(rf, q.reshape(-1), stream), nh * hd,
                            _dev(rf, k.view(np.uint16).reshape(-1), stream), _dev(rf, v.view(np.uint16).reshape(-1), stream),
                            hd, cap * hd, dout, nh * hd)
    finally:
        rf.check(rf.load().rfp4_debug_prefill_ksplit(0))
    got = dout.to_host(rows * nh * hd, np.float32, stream).reshape(rows, nh, hd)
    s = np.einsum("rhd,td->rht", q.astype(np.float64), k.astype(np.float64)) / np.sqrt(hd)
    amp = (np.einsum("rhd,td->rht", abs(q.astype(np.float64)), abs(k.astype(np.float64))) / np.sqrt(hd)).max(-1)
    s[np.broadcast_to(np.arange(cap)[None, None] > pos0 + np.arange(rows)[:, None, None], s.shape)] = -np.inf
    top = np.sort(s, -1)[..., -2:]
    assert np.all(top[..., 1] - top[..., 0] > 2.0 ** -18 * amp) and amp.min() > 70 * 2 ** 19
    np.testing.assert_array_equal(got, v.astype(np.float32)[s.argmax(-1)])
