"""The dense GEMMs' workgroup tiles (64 x 64 and 128 x 128, staged through a
ring of LDS chunks) at ragged sizes: rows and columns one past a tile, the
shortest K, and sizes on either side of each tile's threshold.  Products
whose K is split in quarters keep the small kernels' summation order, so
their rows equal those kernels' rows bit for bit; every product is also
within the dense tolerance of float64 (2^-16 of sum |a b|, plus one bf16
step for bf16 outputs)."""
import numpy as np
import pytest

from helpers import W, host, stream, torch

pytestmark = pytest.mark.gpu


def matrix(seed, rows, columns, sigma):
    t = torch()
    g = t.Generator(device="cuda").manual_seed(seed)
    return (t.randn(rows, columns, generator=g, device="cuda") * sigma).to(t.bfloat16)


def gemm(q38m, a, b, bf16):
    t = torch()
    out = t.empty(a.shape[0], b.shape[0], device="cuda", dtype=t.bfloat16 if bf16 else t.float32)
    q38m.call("q38m_dense_gemm_bf16", a.data_ptr(), b.data_ptr(), a.shape[0], b.shape[0],
              a.shape[1], None if bf16 else out.data_ptr(), out.data_ptr() if bf16 else None,
              stream(), 0)
    return out


def assert_close(got, a, b, bf16):
    ad, bd = a.double(), b.double()
    want = ad @ bd.t()
    bound = 2.0 ** -16 * (ad.abs() @ bd.abs().t()) + (2.0 ** -8 * want.abs() if bf16 else 0.0)
    assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", [(1537, 512, 2048), (12161, 512, 2048), (1500, 500, 1280),
                                   (6209, 1000, 2304)])
def test_split_tiles_equal_small_kernels(q38m, m, n, k, bf16):
    a, b = matrix(m, m, k, 1.0), matrix(n, n, k, 0.02)
    got = gemm(q38m, a, b, bf16)
    for rows in (slice(0, 100), slice(m - 100, m)):
        assert torch().equal(got[rows], gemm(q38m, a[rows].contiguous(), b, bf16))
    assert_close(got, a, b, bf16)


@pytest.mark.parametrize("m,n,k", [(193, 4097, 192), (513, 2048, 512), (6145, 1025, 320),
                                   (12289, 513, 1024), (513, 2048, 160)])
def test_whole_k_tiles(q38m, m, n, k):
    a, b = matrix(m, m, k, 1.0), matrix(n, n, k, 0.04)
    assert_close(gemm(q38m, a, b, True), a, b, True)
    assert_close(gemm(q38m, a, b, False), a, b, False)


@pytest.mark.parametrize("tokens", [801, 6101])
def test_shared_expert_tiles(q38m, tokens):
    t = torch()
    inter = W.INTER
    x = matrix(1, tokens, W.HIDDEN, 1.0)
    wg, wu = matrix(2, inter, W.HIDDEN, 0.02), matrix(3, inter, W.HIDDEN, 0.02)
    wd, wo = matrix(4, W.HIDDEN, inter, 0.04), matrix(5, 1, W.HIDDEN, 0.02)

    def run(rows):
        n = rows.shape[0]
        scratch = t.empty(3, n, inter, dtype=t.bfloat16, device="cuda")
        assert scratch.numel() * 2 == q38m.lib().q38m_moe_shared_expert_scratch_bytes(n, inter)
        out = t.empty(n, W.HIDDEN, dtype=t.bfloat16, device="cuda")
        gate = t.empty(n, dtype=t.bfloat16, device="cuda")
        q38m.call("q38m_moe_shared_expert_v1", rows.data_ptr(), wg.data_ptr(), wu.data_ptr(),
                  wd.data_ptr(), wo.data_ptr(), n, W.HIDDEN, inter, scratch.data_ptr(),
                  out.data_ptr(), gate.data_ptr(), stream(), 0)
        return scratch, out, gate

    scratch, out, gate = run(x)
    for rows in (slice(0, 40), slice(tokens - 40, tokens)):
        small, _, small_gate = run(x[rows].contiguous())
        assert t.equal(scratch[:, rows], small)  # g, u and h
        assert t.equal(gate[rows], small_gate)
    assert_close(out, scratch[2], wd, True)
    assert np.isfinite(host(out.view(t.int16), np.uint16).astype(np.float32)).all()
