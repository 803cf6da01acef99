"""The load path at the edges of its kernels: the W4 repack (one row tile of up
to 16 quads per workgroup) at one quad, a ragged and a second block of quads,
against a numpy statement of the layouts; the quantiser's row kernels (512,
2,048 and other widths) and its group kernels' last piece, with infinite and
NaN weights and with scales that take the division, against the oracle."""
import numpy as np
import pytest

from helpers import device, host, torch
from test_gpu_quantizer import quantize_on_gpu

pytestmark = pytest.mark.gpu


def w4_layout(data, scales, paired):
    """Row-major [E][R][K/2] and [E][R][K/g] -> the quad-major layout."""
    experts, rows, half = data.shape
    quads, tiles = half // 64, rows // 16
    nib = np.stack((data & 15, data >> 4), axis=-1).reshape(experts, rows, quads, 4, 4, 8)
    out = nib[..., :4] | (nib[..., 4:] << 4)             # [E][R][quad][j][q][4 bytes]
    out = out.reshape(experts, tiles, 16, quads, 4, 4, 4)
    out = out.transpose(0, 3, 1, 5, 2, 4, 6)             # [E][quad][tile][q][n][j][byte]
    words = scales.reshape(experts, tiles, 16, quads, -1).transpose(0, 3, 1, 2, 4)
    if paired:
        order = [s // 2 + (s % 2) * tiles // 2 for s in range(tiles)]
        out, words = out[:, :, order], words[:, :, order]
    return np.ascontiguousarray(out).ravel(), np.ascontiguousarray(words).ravel()


@pytest.mark.parametrize("paired", [False, True])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("experts,rows,columns", [(3, 32, 128), (2, 64, 1152), (1, 96, 4480)])
def test_w4_repack_layout(q38m, experts, rows, columns, group, paired):
    t = torch()
    rng = np.random.default_rng(columns + group)
    data = rng.integers(0, 256, (experts, rows, columns // 2), dtype=np.uint8)
    scales = rng.integers(0, 65536, (experts, rows, columns // group), dtype=np.uint16)
    src = q38m.DeviceWeights(device(data), device(scales), q38m.FORMAT_W4_SYM, group,
                             q38m.LAYOUT_ROW_MAJOR, experts, rows, columns)
    dst = q38m.repack(src, paired=paired)
    t.cuda.synchronize()
    want_data, want_scales = w4_layout(data, scales, paired)
    assert np.array_equal(host(dst.data, np.uint8).ravel(), want_data)
    assert np.array_equal(host(dst.scales, np.uint16).ravel(), want_scales)


@pytest.mark.parametrize("bits,group,columns", [(8, 0, 512), (8, 0, 2048), (8, 0, 1536),
                                                (4, 32, 96), (4, 128, 384), (8, 64, 192),
                                                (8, 32, 2048)])
def test_quantizer_edges(q38m, orc, bits, group, columns):
    experts, rows = 1, 37
    rng = np.random.default_rng(columns + bits)
    w = (rng.standard_normal((experts * rows, columns)) *
         rng.choice([1e-38, 1e-3, 0.02, 1e30], (experts * rows, 1))).astype(np.float32)
    w[3, 5], w[4, 9], w[5, :] = np.inf, np.nan, 1e-40
    h = orc.f32_to_bf16(w)
    fmt = q38m.FORMAT_W4_SYM if bits == 4 else q38m.FORMAT_W8_SYM
    data, scales = quantize_on_gpu(q38m, device(h), fmt, group, experts, rows, columns, True)
    want_data, want_scales = orc.quantize_weights(h, bits, group, True)
    assert np.array_equal(host(data, np.uint8).reshape(want_data.shape), want_data)
    assert np.array_equal(host(scales, np.uint16).reshape(want_scales.shape), want_scales)
