"""The slab plan of up to 640 routes (64 tokens), one route per thread, at the
edges of its waves (64 routes), of its expert threads (512) and of its range,
byte for byte against the oracle's plan; 65 tokens take the general kernel."""
import numpy as np
import pytest

from test_gpu_primitives import reference_pattern, run_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 6, 7, 51, 52, 63, 64, 65])
@pytest.mark.parametrize("kind", ["distinct", "all", "random", "invalid"])
def test_small_plan_bitwise(q38m, orc, tokens, kind):
    rng = np.random.default_rng(tokens)
    if kind == "distinct":
        ids = reference_pattern(tokens, None)
    elif kind == "all":
        ids = reference_pattern(tokens, "all")
    else:  # any ids, repeats among them; with some out of range
        ids = rng.integers(0, 512, tokens * 10).astype(np.int32)
        if kind == "invalid":
            ids[rng.integers(0, ids.size, 1 + tokens // 4)] = rng.choice([-1, 512, 1 << 30, -(1 << 31)])
    got = run_plan(q38m, ids, tokens, True, poison=0xA5)
    assert np.array_equal(got, orc.build_plan(ids, tokens, hashes=True))
