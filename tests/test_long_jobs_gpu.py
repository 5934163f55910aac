"""The persistent encoder on jobs past the in-kernel exchange (more than 256
tiles): below and above one round of its grid, a partial last tile, both
quantizers, relative and absolute bounds, a job whose staging overflows, and
a give-up forced from the host.  Streams and bounds against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def store_and_check(oracle, w, pages, eps, relative, quantizer):
    count, n = pages.shape
    bufs = [torch.empty(8 * n, dtype=torch.uint8, device="cuda") for _ in range(count)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16(list(pages), bufs, [eps] * count)
    assert ok
    host = bits(pages)
    for i in range(count):
        eb = np.float32(oracle.relative_bound(host[i], n, eps) if relative else eps)
        assert np.float32(bounds[i]) == eb
        want = oracle.compress_page(host[i], n, float(eb), variant=quantizer)
        assert sizes[i] == len(want)
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want), i


def wrapper(relative, quantizer=0):
    import cuszp_wrapper_cpp as cpp

    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, relative, cpp.DIM_1D, cpp.MODE_FIXED,
                                               cpp.TYPE_FLOAT), 0)
    w.set_codec_options(quantizer, 1)
    return w


def pages_of(count, n, off=0):
    g = torch.Generator().manual_seed(n)
    flat = torch.randn(off + count * n, generator=g).to(torch.bfloat16).cuda()
    return flat[off:].view(count, n)


@pytest.mark.parametrize("count,n,off,relative,quantizer", [
    (1, 256 * 8192 + 32, 0, True, 0),        # 257 tiles, the last of one block
    (2, 300 * 8192, 1, True, 1),
    (2, 777 * 8192 + 4096, 0, True, 0),      # 1556 tiles: past one round
    (1, 1700 * 8192 + 64, 3, False, 0),      # one job longer than the grid
    (5, 257 * 8192, 0, False, 1),
])
def test_long_jobs(oracle, count, n, off, relative, quantizer):
    pages = pages_of(count, n, off)
    pages[0, -1] = 30.0
    store_and_check(oracle, wrapper(relative, quantizer), pages, 1e-4 if relative else 1e-3,
                    relative, quantizer)


def test_overflow_and_uniform(oracle):
    n = 260 * 8192
    pages = pages_of(3, n)
    pages[1] = 1.3125                 # one value: repeated blocks at rate 31
    pages[2, 5] = 3e38                # next to it everything else is rate 0
    w = wrapper(True)
    store_and_check(oracle, w, pages, 1e-4, True, 0)
    w = wrapper(False)                # rates far above 15: encoded again
    before = w._ctx.reencode_count()
    store_and_check(oracle, w, pages_of(2, n) * 1000, 1e-6, False, 0)
    assert w._ctx.reencode_count() == before + 1


MANY = 4096 * 8192   # 8192 tiles in two jobs: more than five rounds of the grid


def until_give_up(ctx, call):
    """Calls until a launch gives up: with a wait bound of zero the first wait
    that is not met at its first poll does, which any of thousands can be."""
    before = ctx.reencode_count()
    for _ in range(5):
        call()
        if ctx.reencode_count() > before:
            break
    assert ctx.reencode_count() == before + 1


def test_give_up(oracle):
    w = wrapper(True)
    w._ctx.set_wait_bound(0)
    store_and_check(oracle, w, pages_of(2, 900 * 8192), 1e-4, True, 0)
    w = wrapper(True)
    w._ctx.set_wait_bound(0)
    pages = pages_of(2, MANY)
    until_give_up(w._ctx, lambda: store_and_check(oracle, w, pages, 1e-4, True, 0))
