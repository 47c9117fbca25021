"""Prompts one after another through one engine (its prompt buffer is reused
and regrown: 1, 256 and 257 tokens around a growth) against a new engine for
each: the same token, logits and K/V."""
import numpy as np
import pytest

from test_gpu_prefill import TINY, _engine

pytestmark = pytest.mark.gpu


def test_prompts_in_turn(rf):
    cfg = dict(TINY, max_seq=600)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, cfg["vocab"], n).astype(np.uint32) for n in (1, 256, 255, 257, 3, 256)]
    eng = _engine(rf, cfg, 9)
    for p in prompts:
        tok, logits = eng.prefill(p, 0), eng.logits()
        new = _engine(rf, cfg, 9)
        assert new.prefill(p, 0) == tok
        np.testing.assert_array_equal(new.logits(), logits)
        assert int(np.argmax(logits)) == tok
