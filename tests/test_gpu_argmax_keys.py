"""The reduction of an argmax GEMV's per-workgroup keys (rfp4_argmax_keys):
key counts around its 1024 threads and its four loads per thread, ties and
NaN logits, against numpy on the logits that the same call returns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one 32-value block per row; 8 rows per key below 16384 rows, 32 from there on
@pytest.mark.parametrize("n", [1, 8, 9, 8 * 1023 + 1, 8 * 1024, 8 * 1025, 32 * 1025, 32 * 4097 + 1])
def test_argmax_keys(rf, stream, n):
    k = 32
    rng = np.random.default_rng(n)
    codes = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    scales = np.full((n, 1), 120, dtype=np.uint8)
    # the row of the largest logit three times, a NaN row in front of it
    x = rng.standard_normal(k).astype(np.float32)
    lut = np.array([0, .5, 1, 1.5, 2, 3, 4, 6], np.float32)
    best = np.where(x > 0, 7, 15).astype(np.uint8)  # +-6 along x: above every other row
    assert lut[7] == 6
    row = best[0::2] | (best[1::2] << 4)
    at = sorted({n // 3, n // 2, n - 1})
    codes[at] = row
    if n > 2:
        scales[0] = 255  # E8M0 NaN
        at = [i for i in at if i > 0]
    bufs = [rf.DeviceBuffer.from_host(a, stream) for a in (codes, scales, x)]
    y = rf.DeviceBuffer.zeroed(n, np.float32, stream)
    ws = rf.DeviceBuffer(rf.mx4_gemv_argmax_workspace(n))
    tok = rf.DeviceBuffer.zeroed(1, np.uint32, stream)
    for _ in range(3):  # the workspace holds the previous call's keys
        rf.mx4_gemv_argmax(stream, n, k, *bufs, y, ws, tok)
    logits = y.to_host(n, np.float32, stream)
    got = int(tok.to_host(1, np.uint32, stream)[0])
    assert got == at[0] == int(np.nanargmax(logits))
