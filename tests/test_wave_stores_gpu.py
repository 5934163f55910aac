"""The BF16 decoders' wave-wide stores: destinations at any 2-byte address,
runs that end inside a wave, layers and destinations that change inside one,
rate-0 blocks written or skipped.  Values against the oracle, and nothing
outside the destinations touched."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import fixed_wrapper

pytestmark = pytest.mark.gpu

FILL = 1.75


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def stored(w, n, seed):
    """(streams, sizes, bounds) of three segments of n values, a third of the
    first in rate-0 blocks."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(3, n, generator=g)
    x[0, : n // 3] = 0.0
    cap = max(8 * n, 1024 * -(-n // 32768) + 128 * -(-n // 32))
    bufs = [torch.empty(cap, dtype=torch.uint8, device="cuda") for _ in range(3)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16(
        list(x.to(torch.bfloat16).cuda()), bufs, [1e-4, 1e-3, 1e-5])
    assert ok
    return bufs, sizes, bounds


def host(bufs, sizes):
    return [b[:s].cpu().numpy() for b, s in zip(bufs, sizes)]


@pytest.mark.parametrize("rate0", [0, 1])
@pytest.mark.parametrize("n,off", [(33, 1), (2047, 0), (2049, 5), (8192 + 2048, 1),
                                   (2 * 8192 - 31, 3), (700 * 8192 + 33, 1)])
def test_linear(oracle, n, off, rate0):
    # 3 x 701 tiles: past the persistent decoder's 2048 workgroups
    w = fixed_wrapper()
    w.set_codec_options(0, rate0)
    bufs, sizes, bounds = stored(w, n, n)
    out = torch.full((off + 3 * n + 9,), FILL, dtype=torch.bfloat16, device="cuda")
    want = bits(out)
    assert w.decompress_batch_fixed_bf16(bufs, sizes, out[off:], n, bounds)
    assert w.synchronize()
    for i, s in enumerate(host(bufs, sizes)):
        lo = off + i * n
        want[lo:lo + n] = oracle.decompress_contiguous(s, n, bounds[i], rate0,
                                                       want[lo:lo + n].copy())
    assert np.array_equal(bits(out), want)


@pytest.mark.parametrize("rate0", [0, 1])
@pytest.mark.parametrize("dpp,epd,off", [(2, 4096, 1), (3, 2080, 0), (4, 6400, 0), (5, 333, 3)])
def test_destinations(oracle, dpp, epd, off, rate0):
    w = fixed_wrapper()
    w.set_codec_options(0, rate0)
    n = dpp * epd
    bufs, sizes, bounds = stored(w, n, n)
    step = epd + off + 7
    slab = torch.full((3 * dpp * step,), FILL, dtype=torch.bfloat16, device="cuda")
    dests = [slab[k * step + off:k * step + off + epd] for k in range(3 * dpp)]
    want = bits(slab)
    assert w.decompress_batch_fixed_bf16_scatter(bufs, sizes, dests, n, dpp, epd, bounds)
    assert w.synchronize()
    for i, s in enumerate(host(bufs, sizes)):
        parts = [want[k * step + off:k * step + off + epd].copy()
                 for k in range(i * dpp, (i + 1) * dpp)]
        oracle.decompress_scatter(s, n, bounds[i], parts, epd, rate0)
        for k, part in zip(range(i * dpp, (i + 1) * dpp), parts):
            want[k * step + off:k * step + off + epd] = part
    assert np.array_equal(bits(slab), want)


@pytest.mark.parametrize("rate0", [0, 1])
@pytest.mark.parametrize("prefix,src,epl,idx,off", [
    (2, 5, 6400, [4, 0, 3], 0),       # layers of 3.125 waves
    (2, 4, 32 * 7, [1, 3, 0], 1),     # many layers in a wave, odd addresses
    (3, 3, 2048 * 3 + 40, [2, 0], 0),  # blocks straddle layers
])
def test_layers(oracle, prefix, src, epl, idx, off, rate0):
    w = fixed_wrapper()
    w.set_codec_options(0, rate0)
    n = prefix * len(idx) * epl
    bufs, sizes, bounds = stored(w, n, n)
    page = prefix * src * epl
    slab = torch.full((off + 3 * page + 9,), FILL, dtype=torch.bfloat16, device="cuda")
    dests = [slab[off + i * page:off + (i + 1) * page] for i in range(3)]
    want = bits(slab)
    assert w.decompress_batch_fixed_bf16_indexed_scatter(
        bufs, sizes, dests, torch.tensor(idx, device="cuda"), prefix, src, epl, bounds)
    assert w.synchronize()
    for i, s in enumerate(host(bufs, sizes)):
        part = want[off + i * page:off + (i + 1) * page].copy()
        oracle.decompress_indexed(s, n, bounds[i], part, idx, src, epl, rate0)
        want[off + i * page:off + (i + 1) * page] = part
    assert np.array_equal(bits(slab), want)
