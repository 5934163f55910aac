"""fp32 pages encoded in one pass: the bound exchanged between a page's tiles
inside the kernel (1 to 256 tiles; one more takes the pre-pass), wave-wide
loads at any 4-byte address, payloads through LDS and, past what that holds
(rates above 15), straight from the lanes.  NaN, infinities, zeros and one-sign
pages, a give-up forced from the host.  Streams, sizes, bounds against the
oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = 8


def pages_of(n, off):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(KINDS, n, generator=g)
    x[0, -1] = 50.0
    x[1] = x[1].abs() + 0.5
    x[2] = -x[2].abs()
    x[3] = 0.0
    x[3, 0] = -0.0
    x[4, n // 2] = float("nan")
    x[5, 0], x[5, -1] = float("inf"), -2.0
    x[6] = 1.7
    x[7, : n // 2] = 0.0
    flat = torch.zeros(off + x.numel(), device="cuda")
    flat[off:] = x.flatten().cuda()
    return flat[off:].view(KINDS, n)


def same_bound(a, b):
    a, b = np.float32(a), np.float32(b)
    return a == b or (np.isnan(a) and np.isnan(b))


@pytest.mark.parametrize("mode", ["fixed", "plain", "outlier"])
@pytest.mark.parametrize("n,off,eps", [(1, 1, 1e-4), (2047, 0, 1e-4), (2048, 3, 1e-7),
                                       (8192 + 33, 1, 1e-3), (28 * 8192, 0, 1e-4),
                                       (5 * 8192 + 2048, 2, 3e-6)])
def test_modes(oracle, mode, n, off, eps):
    import cuszp_wrapper_cpp as cpp

    m = {"fixed": cpp.MODE_FIXED, "plain": cpp.MODE_PLAIN, "outlier": cpp.MODE_OUTLIER}[mode]
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, True, cpp.DIM_1D, m, cpp.TYPE_FLOAT), 0)
    pages = pages_of(n, off)
    host = pages.cpu().numpy()
    for i in range(KINDS):
        buf = torch.full((8 * n + 1024 + 136,), 0xAB, dtype=torch.uint8, device="cuda")
        ok, buf, size, bound = w.compress(pages[i], buf, eps)
        assert ok
        eb = oracle.relative_bound_f32(host[i], eps)
        assert same_bound(bound, eb), i
        want = (oracle.compress_page_f32(host[i], float(eb)) if mode == "fixed"
                else oracle.compress_page_f32_mode(host[i], float(eb), int(m)))
        assert size == want.size, i
        assert np.array_equal(buf[:size].cpu().numpy(), want), i
        assert bool((buf[size:] == 0xAB).all()), i


@pytest.mark.parametrize("n", [255 * 8192 + 64, 256 * 8192, 256 * 8192 + 1])
@pytest.mark.parametrize("give_up", [False, True])
def test_batches(oracle, n, give_up):
    import cuszp_wrapper_cpp as cpp

    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, True, cpp.DIM_1D, cpp.MODE_FIXED,
                                               cpp.TYPE_FLOAT), 0)
    if give_up:
        w._ctx.set_wait_bound(0)
    pages = pages_of(n, 0)[:3]
    bufs = [torch.empty(8 * n, dtype=torch.uint8, device="cuda") for _ in range(3)]
    before = w._ctx.reencode_count()
    ok, sizes, bounds = w.compress_batch_fixed(list(pages), bufs, [1e-4, 1e-3, 1e-5])
    assert ok
    # past 256 tiles the pre-pass gives the bound and no wait is timed
    assert w._ctx.reencode_count() - before == (1 if give_up and n <= 256 * 8192 else 0)
    for i, eps in enumerate((1e-4, 1e-3, 1e-5)):
        x = pages[i].cpu().numpy()
        eb = oracle.relative_bound_f32(x, eps)
        assert same_bound(bounds[i], eb)
        want = oracle.compress_page_f32(x, float(eb))
        assert sizes[i] == want.size
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want), i
