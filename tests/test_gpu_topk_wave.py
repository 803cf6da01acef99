"""The top-10 of large calls, one wave per token, against the small calls'
ten-wave workgroups, bit for bit: ragged counts from the rule's line on, ties,
infinities, NaN of both signs and rows of one value."""
import numpy as np
import pytest

from helpers import host, stream, synth_logits, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1280, 1283, 4099])
def test_wave_topk_equals_block_topk(q38m, tokens):
    t = torch()
    logits = synth_logits(q38m, 5, 6, tokens).clone()
    logits[7] = 0.25
    logits[8] = t.round(logits[8])  # ties
    logits[9, ::3] = float("inf")
    logits[10] = float("-inf")
    logits[11, 5:300] = float("nan")
    logits[12] = -logits[11]
    logits[13] = t.finfo(t.float32).min
    logits[14] = t.where(t.arange(512, device="cuda") % 2 == 0, 0.0, -0.0)
    logits[tokens - 1, 100:105] = float("inf")

    def run(first, count):
        ids = t.full((count, 10), -7, dtype=t.int32, device="cuda")
        weights = t.full((count, 10), -7.0, device="cuda")
        part = logits[first:first + count].contiguous()
        q38m.call("q38m_topk_router_f32", part.data_ptr(), ids.data_ptr(), weights.data_ptr(),
                  count, 512, 10, 1, stream(), 0)
        return host(ids, np.int32), host(weights, np.uint32)

    ids, weights = run(0, tokens)
    for first in range(0, tokens, 512):
        count = min(512, tokens - first)
        want_ids, want_weights = run(first, count)
        rows = slice(first * 10, (first + count) * 10)
        assert np.array_equal(ids.ravel()[rows], want_ids.ravel())
        assert np.array_equal(weights.ravel()[rows], want_weights.ravel())
