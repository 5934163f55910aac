"""Rates that fill the persistent encoder's staging words: blocks of 16 to 24
planes are encoded in one launch in each of its kinds, blocks of 25 planes
throughout are marked and encoded again.  Streams against the oracle, and the
context's count of second encodes."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# kind: values of a segment, offset from an aligned address, layers of its page
KINDS = {
    "plain": (3 * 8192, 0, None),
    "odd address": (3 * 8192, 1, None),
    "cut": (3 * 8192 + 95, 1, None),
    "split": (2 * 2 * 6400, 0, (2, 5, 6400, [4, 1])),
    "long": (257 * 8192, 0, None),
}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("rate", [16, 24, 25])
def test_rates(oracle, kind, rate):
    import cuszp_wrapper_cpp as cpp

    n, off, layers = KINDS[kind]
    numel = layers[0] * layers[1] * layers[2] if layers else n
    g = torch.Generator().manual_seed(rate)
    # magnitudes in [1, 2) on both sides: with eb = 2^-rate every |q| lies in
    # [2^(rate - 1), 2^rate)
    x = (1 + torch.rand(off + 2 * numel, generator=g) * 0.99)
    x *= torch.randint(0, 2, x.shape, generator=g) * 2 - 1
    pages = x.to(torch.bfloat16).cuda()[off:].view(2, numel)
    eps = 2.0 ** -rate
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(eps, False, cpp.DIM_1D, cpp.MODE_FIXED,
                                               cpp.TYPE_FLOAT), 0)
    cap = max(8 * n, 1024 * -(-n // 32768) + 128 * -(-n // 32))
    bufs = [torch.full((cap,), 0xAB, dtype=torch.uint8, device="cuda") for _ in range(2)]
    before = w._ctx.reencode_count()
    if layers:
        prefix, src, epl, idx = layers
        ok, sizes, _ = w.compress_batch_fixed_bf16_indexed(
            list(pages), bufs, torch.tensor(idx, device="cuda"), prefix, src, epl, [eps] * 2)
    else:
        src, epl, idx = 0, 0, None
        ok, sizes, _ = w.compress_batch_fixed_bf16(list(pages), bufs, [eps] * 2)
    assert ok
    assert w._ctx.reencode_count() - before == (1 if rate > 24 else 0)
    host = pages.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
    for i in range(2):
        want = oracle.compress_page(host[i], n, eps, idx, src, epl)
        assert sizes[i] == len(want)
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want), i
        assert bool((bufs[i][sizes[i]:] == 0xAB).all()), i
