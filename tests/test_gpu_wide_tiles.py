"""The chunk path's 32x32 MFMA kernels (groups of 64 and 128, W8 per channel
gate/up) at the edges of their row tiles: experts of 1 to 129 routes (one row,
one short of and one past the 32-row tiles, the 64-row workgroups and the
128-row tasks).  At T <= 512 the chunk plan's packed order is the slab's, so
every mid word and route output must equal the slab path's bit for bit (the
slab path is pinned to the oracle in test_gpu_formats.py)."""
import numpy as np
import pytest

from helpers import Layer, host, prefill, synth_hidden, synth_logits, torch, ws_arrays
from test_gpu_wide import prefill_wide

pytestmark = pytest.mark.gpu

ROWS = (1, 31, 33, 63, 65, 95, 97, 127, 129)
FORMATS = {
    "w4g64bf16-w4g128": (((4, 64, 0.02), True), ((4, 128, 0.02), False)),
    "w4g128-w4g64bf16": (((4, 128, 0.02), False), ((4, 64, 0.02), True)),
    "w8g64-w8g128bf16": (((8, 64, 0.002), False), ((8, 128, 0.002), True)),
    "w8pcbf16-w8g64": (((8, 0, 0.002), True), ((8, 64, 0.002), False)),
    "w8g128bf16-w8g128": (((8, 128, 0.002), True), ((8, 128, 0.002), False)),
}


@pytest.mark.parametrize("name", list(FORMATS))
def test_row_tile_edges_equal_slab(q38m, orc, name):
    (gfmt, gbf16), (dfmt, dbf16) = FORMATS[name]
    layer = Layer(q38m, orc, 17, 5, ("fmt",) + gfmt, ("fmt",) + dfmt, with_host=False,
                  gate_up_bf16=gbf16, down_bf16=dbf16)
    tokens = 200
    hidden = synth_hidden(q38m, 17, 71, tokens)
    logits = synth_logits(q38m, 17, 72, tokens)
    for k, rows in enumerate(ROWS):  # experts 3, 60, 117, ...: the first `rows` tokens
        logits[:, 3 + 57 * k] = -40.0
        logits[:rows, 3 + 57 * k] = 30.0 + k
    slab, chunk = q38m.PrefillWorkspace_(tokens), q38m.WideWorkspace_(tokens)
    out_slab = prefill(q38m, layer, hidden, logits, slab)
    out_chunk = prefill_wide(q38m, layer, hidden, logits, chunk)
    a, b = ws_arrays(slab, tokens), ws_arrays(chunk, tokens)
    counts = np.bincount(a["ids"].ravel(), minlength=512)
    assert tuple(counts[3 + 57 * k] for k in range(len(ROWS))) == ROWS
    assert np.array_equal(a["weighted_mid"], b["weighted_mid"])
    assert np.array_equal(a["route_output"].view(np.uint32), b["route_output"].view(np.uint32))
    assert np.array_equal(host(out_slab, np.uint16), host(out_chunk, np.uint16))
    torch().cuda.empty_cache()
