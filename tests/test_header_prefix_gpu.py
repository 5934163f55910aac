"""Tile offsets of the one-workgroup-per-tile decoders: jobs of 1, 64 and 65
tiles (header sums up to 64 tiles, look-back beyond), in every encoding mode
and as BF16, rate-0 blocks and outlier words among the header bytes.  Values
against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import fixed_wrapper

pytestmark = pytest.mark.gpu

SIZES = [8192, 2 * 8192 + 5, 64 * 8192, 64 * 8192 + 1]


def values(n):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g).cumsum(0) * 0.05   # smooth: small residuals
    x[n // 3: n // 2] = 0.0
    x[-40:] = 3.0
    return x


@pytest.mark.parametrize("mode", ["fixed", "plain", "outlier"])
@pytest.mark.parametrize("n", SIZES)
def test_fp32(oracle, mode, n):
    import cuszp_wrapper_cpp as cpp

    m = {"fixed": cpp.MODE_FIXED, "plain": cpp.MODE_PLAIN, "outlier": cpp.MODE_OUTLIER}[mode]
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, True, cpp.DIM_1D, m, cpp.TYPE_FLOAT), 0)
    buf = torch.empty(8 * n + 2048, dtype=torch.uint8, device="cuda")
    ok, buf, size, bound = w.compress(values(n).cuda(), buf, 1e-4)
    assert ok
    stream = buf[:size].cpu().numpy()
    want = (oracle.decompress_f32(stream, n, bound) if mode == "fixed"
            else oracle.decompress_f32_mode(stream, n, bound, int(m)))
    out = torch.full((n,), 5.5, device="cuda")
    assert w.decompress(buf, size, out, bound)
    assert w.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n", SIZES)
def test_bf16(oracle, n):
    w = fixed_wrapper()
    x = values(n).to(torch.bfloat16).cuda()
    buf = torch.empty(8 * n, dtype=torch.uint8, device="cuda")
    ok, sizes, bounds = w.compress_batch_fixed_bf16([x], [buf], [1e-4])
    assert ok
    out = torch.full((n,), 5.5, dtype=torch.bfloat16, device="cuda")
    assert w.decompress_batch_fixed_bf16([buf], sizes, out, n, bounds)
    assert w.synchronize()
    want = oracle.decompress_contiguous(buf[:sizes[0]].cpu().numpy(), n, bounds[0])
    got = out.view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(got, want)
