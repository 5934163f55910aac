"""The fp32 decoders' wave-wide stores: segments that end inside a wave's run
or just past it, outputs at any 4-byte address, rate-0 blocks written or
skipped.  Values against the oracle, and nothing outside the output touched."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fixed", "plain", "outlier"])
@pytest.mark.parametrize("n,off", [(31, 1), (2047, 0), (2048, 1), (2049, 3), (8192 + 2048, 2),
                                   (3 * 8192 - 32, 1)])
@pytest.mark.parametrize("rate0", [0, 1])
def test_fp32_wave_stores(oracle, mode, n, off, rate0):
    import cuszp_wrapper_cpp as cpp

    m = {"fixed": cpp.MODE_FIXED, "plain": cpp.MODE_PLAIN, "outlier": cpp.MODE_OUTLIER}[mode]
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, True, cpp.DIM_1D, m, cpp.TYPE_FLOAT), 0)
    w.set_codec_options(0, rate0)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g)
    x[: n // 3] = 0.0                                # rate-0 blocks
    buf = torch.empty(8 * n + 1024 + 136, dtype=torch.uint8, device="cuda")
    ok, buf, size, bound = w.compress(x.cuda(), buf, 1e-3)
    assert ok
    stream = buf[:size].cpu().numpy()
    if mode == "fixed":
        want = oracle.decompress_f32(stream, n, bound)
    else:
        want = oracle.decompress_f32_mode(stream, n, bound, int(m))
    slab = torch.full((off + n + 64,), 5.5, device="cuda")
    assert w.decompress_batch([buf], [size], [slab[off:off + n]], [bound])
    assert w.synchronize()
    got = slab.cpu().numpy()
    out = got[off:off + n]
    skipped = np.zeros(n, bool)
    if not rate0:  # blocks whose header byte is 0 stay as they were
        skipped = np.repeat(stream[: -(-n // 32)] == 0, 32)[:n]
        assert skipped.any() or n < 96
    assert np.array_equal(out[~skipped].view(np.uint32), want[~skipped].view(np.uint32))
    assert (out[skipped] == 5.5).all()
    assert (got[:off] == 5.5).all() and (got[off + n:] == 5.5).all()
