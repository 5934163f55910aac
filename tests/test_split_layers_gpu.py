"""The persistent encoder on layers that are no whole number of a wave's 2048
values: a run that goes on in the next layer, in the next prefix, in several
short layers, at odd addresses, in both look-back placements (jobs of up to 24
tiles and longer).  Streams and bounds against the oracle; a bad layer index
met only by the second part of a run is reported."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import fixed_wrapper

pytestmark = pytest.mark.gpu


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def pages_of(count, numel, off):
    g = torch.Generator().manual_seed(numel)
    flat = torch.randn(off + count * numel, generator=g).to(torch.bfloat16).cuda()
    return flat[off:].view(count, numel)


@pytest.mark.parametrize("prefix,src,epl,idx,off", [
    (2, 5, 6400, [4, 0, 3], 0),
    (2, 3, 2080, [2, 0], 1),
    (3, 2, 2048 + 1024, [1], 0),       # a single layer: every crossing wraps
    (2, 6, 32 * 7, [5, 0, 3, 1], 3),   # several layers in one run
    (2, 9, 19232, [8, 1, 0, 2, 7, 3, 5, 4, 6], 0),  # 43 tiles a job
])
def test_split_layers(oracle, prefix, src, epl, idx, off):
    pages = pages_of(3, prefix * src * epl, off)
    pages[1] = pages[1].abs()
    n = prefix * len(idx) * epl
    cap = max(8 * n, 1024 * -(-n // 32768) + 128 * -(-n // 32))
    bufs = [torch.empty(cap, dtype=torch.uint8, device="cuda") for _ in range(3)]
    w = fixed_wrapper()
    eps = [1e-4, 1e-3, 1e-5]
    ok, sizes, bounds = w.compress_batch_fixed_bf16_indexed(
        list(pages), bufs, torch.tensor(idx, device="cuda"), prefix, src, epl, eps)
    assert ok
    host = bits(pages)
    for i in range(3):
        eb = oracle.relative_bound(host[i], n, eps[i], idx, src, epl)
        assert np.float32(bounds[i]) == np.float32(eb)
        want = oracle.compress_page(host[i], n, float(eb), idx, src, epl)
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want)


@pytest.mark.parametrize("idx", [[9, 0, 1], [0, 9, 1], [0, 1, -1]])
def test_bad_layer_index(idx):
    prefix, src, epl = 2, 4, 2080
    pages = pages_of(2, prefix * src * epl, 0)
    n = prefix * len(idx) * epl
    bufs = [torch.empty(8 * n, dtype=torch.uint8, device="cuda") for _ in range(2)]
    w = fixed_wrapper()
    ok, _, _ = w.compress_batch_fixed_bf16_indexed(
        list(pages), bufs, torch.tensor(idx, device="cuda"), prefix, src, epl, [1e-4] * 2)
    assert not ok
