"""The hyper-connection prepare above 512 tokens (the low-rank products on
workgroup tiles: K quarters side by side, and the mix-up with its sigmoid and
the stream mix in one kernel): every token equals the same token in a prepare
of up to 512, bit for bit (that sequence is pinned to the oracle in
test_gpu_hyper.py).  Token counts one past a tile, ranks that end in half a
64-wide chunk (the shortest included), both hidden widths, a state with
infinite and NaN values, and hidden widths whose products keep the separate
launches."""
import pytest

from helpers import stream, torch

pytestmark = pytest.mark.gpu


def matrix(g, rows, columns, sigma):
    t = torch()
    return (t.randn(rows, columns, generator=g, device="cuda") * sigma).to(t.bfloat16)


@pytest.mark.parametrize("tokens,hidden,rank,special", [
    (513, 2048, 320, False), (641, 2560, 96, False), (1025, 2048, 32, False),
    (1500, 2048, 288, True), (6500, 2048, 320, False), (520, 1000, 64, False),
    (600, 2080, 128, False)])
def test_large_prepare_equals_small(q38m, tokens, hidden, rank, special):
    assert_prepare_equals_slices(q38m, tokens, hidden, rank, special, 500)


# past the line from which mix-down keeps K in one workgroup (512 tiles of 64 x
# 64: 6,529 tokens at rank 320), and ranks above 1,024 (mix-down without
# partials, mix-up with K split and the sigmoid in its epilogue, a separate
# stream mix); slices of 500 tokens and of 30, whose products run on the
# K-split kernels
@pytest.mark.parametrize("tokens,hidden,rank", [(6600, 2048, 320), (6529, 2560, 320),
                                                (1500, 2048, 1280), (2600, 2560, 1280)])
@pytest.mark.parametrize("count", [500, 30])
def test_prepare_past_the_quarters(q38m, tokens, hidden, rank, count):
    assert_prepare_equals_slices(q38m, tokens, hidden, rank, False, count)


def assert_prepare_equals_slices(q38m, tokens, hidden, rank, special, count):
    t = torch()
    g = t.Generator(device="cuda").manual_seed(tokens)
    wide = 4 * hidden
    state = matrix(g, tokens, wide, 1.0)
    if special:
        state[3, 17], state[600, hidden + 5], state[tokens - 1, 9] = float("inf"), float("nan"), 3e38
    norm = matrix(g, 1, wide, 0.1)
    down, up = matrix(g, rank, wide, wide ** -0.5), matrix(g, wide, rank, 4 * rank ** -0.5)
    inject = matrix(g, 4, wide, wide ** -0.5)

    def run(x):
        n = x.shape[0]
        scratch = t.empty(q38m.lib().q38m_hyper_prepare_scratch_bytes(n, hidden, rank),
                          dtype=t.uint8, device="cuda")
        mixed = t.empty(n, hidden, dtype=t.bfloat16, device="cuda")
        injection = t.empty(n, 4, dtype=t.bfloat16, device="cuda")
        q38m.call("q38m_hyper_prepare_v1", x.data_ptr(), norm.data_ptr(), down.data_ptr(),
                  up.data_ptr(), inject.data_ptr(), n, hidden, rank, scratch.data_ptr(),
                  mixed.data_ptr(), injection.data_ptr(), stream(), 0)
        return mixed, injection

    def words(x):  # every NaN as one word
        return t.where(x.isnan(), t.full_like(x, float("nan")), x).view(t.int16)

    mixed, injection = run(state)
    for rows in (slice(0, count), slice(tokens - count, tokens)):
        small_mixed, small_injection = run(state[rows].contiguous())
        assert t.equal(words(mixed[rows]), words(small_mixed))
        assert t.equal(words(injection[rows]), words(small_injection))
    assert bool(mixed[100:200].isfinite().all()) and mixed[100:200].float().std() > 0.05
