"""Dense products of few rows beside many columns (one to seven row tiles:
columns dealt to the XCDs, or the row tiles spread over them), at ragged sizes
and on either side of the rules that pick a form.  Products whose K is split
give the words of the small kernels, taken over slices of the columns; whole-K
products are within the dense tolerance.  The shared expert over wide
intermediate sizes gives the words of its slices of 512 channels, and the
hyper-connection prepare with one, three and nine channel pairs those of a
prepare of up to 512 tokens."""
import pytest

import test_gpu_hyper_tiles as hyper
from helpers import W, stream, torch
from test_gpu_dense_tiles import assert_close, gemm, matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(2, 16385, 2048), (32, 12290, 2048), (33, 12290, 2048),
                                   (64, 16385, 1280), (65, 25000, 2048), (200, 16385, 2048),
                                   (321, 2049, 2048), (385, 2050, 4096), (577, 6145, 2048),
                                   (1300, 3000, 1280)])
def test_split_products_equal_column_slices(q38m, m, n, k):
    a, b = matrix(m, m, k, 1.0), matrix(n, n, k, 0.02)
    got = gemm(q38m, a, b, False)
    rows = slice(0, m) if m <= 400 else slice(m - 100, m)
    for cols in (slice(0, 70), slice(n // 2, n // 2 + 70), slice(n - 70, n)):
        small = gemm(q38m, a[rows].contiguous(), b[cols].contiguous(), False)
        assert torch().equal(got[rows, cols], small)
    assert_close(got, a, b, False)


@pytest.mark.parametrize("m,n,k", [(2, 40001, 320), (64, 16385, 512), (65, 16385, 1024),
                                   (600, 8193, 768), (1500, 12289, 192), (16385, 70, 320)])
def test_whole_k_products(q38m, m, n, k):
    a, b = matrix(m, m, k, 1.0), matrix(n, n, k, 0.04)
    assert_close(gemm(q38m, a, b, True), a, b, True)
    assert_close(gemm(q38m, a, b, False), a, b, False)


@pytest.mark.parametrize("k,forms", [(192, ((8192, 16385), (4097, 4097), (9000, 16385))),
                                     (320, ((64, 16385), (100, 16385), (700, 16385))),
                                     (512, ((100, 16385), (400, 16385), (530, 12310))),
                                     (1024, ((100, 16385), (400, 16385)))])
def test_whole_k_forms_agree(q38m, k, forms):
    """One accumulator over K in each form: the same words for the rows and
    columns that the sizes share (k 192: the small tiles, 33 x 33 of 128 x 128,
    71 x 129; k 320: the small tiles, 64 x 64, 128 x 128; k 512: 64 x 64, 64 x 64
    where 128 x 128 would be 516 tiles, 128 x 128; k 1,024: 64 x 64, 128 x 128)."""
    t = torch()
    rows, columns = max(m for m, _ in forms), max(n for _, n in forms)
    a, b = matrix(k, rows, k, 1.0), matrix(k + 1, columns, k, 0.04)
    shared_rows, shared_columns = min(m for m, _ in forms), min(n for _, n in forms)
    for bf16 in (False, True):
        results = [gemm(q38m, a[:m], b[:n], bf16)[:shared_rows, :shared_columns] for m, n in forms]
        for other in results[1:]:
            assert t.equal(results[0], other)


@pytest.mark.parametrize("tokens,inter", [(2, 8192), (32, 6144), (33, 6176), (100, 4096), (600, 4128)])
def test_shared_expert_equals_channel_slices(q38m, tokens, inter):
    t = torch()
    x = matrix(1, tokens, W.HIDDEN, 1.0)
    wg, wu = matrix(2, inter, W.HIDDEN, 0.02), matrix(3, inter, W.HIDDEN, 0.02)
    wd, wo = matrix(4, W.HIDDEN, inter, 0.02), matrix(5, 1, W.HIDDEN, 0.02)

    def run(channels):
        n = wg[channels].shape[0]
        parts = [w.contiguous() for w in (wg[channels], wu[channels], wd[:, channels])]
        scratch = t.empty(3, tokens, n, dtype=t.bfloat16, device="cuda")
        out = t.empty(tokens, W.HIDDEN, dtype=t.bfloat16, device="cuda")
        gate = t.empty(tokens, dtype=t.bfloat16, device="cuda")
        q38m.call("q38m_moe_shared_expert_v1", x.data_ptr(), *(w.data_ptr() for w in parts),
                  wo.data_ptr(), tokens, W.HIDDEN, n, scratch.data_ptr(), out.data_ptr(),
                  gate.data_ptr(), stream(), 0)
        return scratch, out, gate

    scratch, out, gate = run(slice(0, inter))
    for channels in (slice(0, 512), slice(inter - 512, inter)):
        small, _, small_gate = run(channels)
        assert t.equal(scratch[:, :, channels], small)  # g, u and h
        assert t.equal(gate, small_gate)
    assert_close(out, scratch[2], wd, True)


@pytest.mark.parametrize("tokens,hidden,rank", [(6500, 32, 32), (2100, 160, 64), (700, 544, 96)])
def test_prepare_of_few_channel_pairs(q38m, tokens, hidden, rank):
    hyper.test_large_prepare_equals_small(q38m, tokens, hidden, rank, False)
