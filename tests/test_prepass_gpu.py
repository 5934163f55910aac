"""The relative-bound pre-pass over segments of every shape it meets: BF16
segments and fp32 pages of more than 256 tiles (up to there the bound is
exchanged inside the encoder, as in test_fp32_pages), in workgroups of one and
of several tiles.  The extremes sit where a wave's wide loads end (a partial
last run or block), at the ends of neighbouring jobs, and at addresses that are
only 2- or 4-byte aligned.  Bounds and streams against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import fixed_wrapper

pytestmark = pytest.mark.gpu

LONG = 256 * 8192  # the longest exchange; one more tile takes the pre-pass


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def flat_pages(count, n, off, dtype, seed):
    """`count` pages of n values one behind the other, `off` values past an
    aligned address."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(off + count * n, generator=g).to(dtype).cuda()
    return x[off:].view(count, n)


def buffer(n):
    cap = 1024 * -(-n // 32768) + 136 * -(-n // 32)
    return torch.empty(max(8 * n, cap), dtype=torch.uint8, device="cuda")


@pytest.mark.parametrize("n,off", [(LONG + 1, 0), (LONG + 2047, 1), (LONG + 2048, 7),
                                   (LONG + 8192 - 31, 3)])
def test_long_bf16(oracle, n, off):
    pages = flat_pages(2, n, off, torch.bfloat16, n)
    pages[0, -1], pages[0, 0] = 9.0, -11.0       # the extremes at both ends
    pages[1] = pages[1].abs()                     # one sign: the general keys
    pages[1, n - 1 - n % 32] = float("nan")
    w = fixed_wrapper()
    bufs = [buffer(n) for _ in range(2)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16(list(pages), bufs, [1e-4, 1e-3])
    assert ok
    host = bits(pages)
    for i, eps in enumerate((1e-4, 1e-3)):
        eb = oracle.relative_bound(host[i], n, eps)
        assert np.float32(bounds[i]) == np.float32(eb)
        want = oracle.compress_page(host[i], n, float(eb))
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want)


def test_long_bf16_runs_across_layers(oracle):
    """Layers of an odd multiple of 32 values: waves' runs straddle them."""
    epl, src, idx = 32 * 22001, 4, [3, 0]
    pages = flat_pages(2, 2 * src * epl, 0, torch.bfloat16, 3)
    view = pages.view(2, 2, src, epl)
    view[0, 1, 0, -1], view[0, 0, 1, 5] = 8.0, 50.0   # selected and unselected layer
    n = 2 * len(idx) * epl
    w = fixed_wrapper()
    bufs = [buffer(n) for _ in range(2)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16_indexed(
        list(pages), bufs, torch.tensor(idx, device="cuda"), 2, src, epl, [1e-4] * 2)
    assert ok
    host = bits(pages)
    for i in range(2):
        eb = oracle.relative_bound(host[i], n, 1e-4, idx, src, epl)
        assert np.float32(bounds[i]) == np.float32(eb)
        want = oracle.compress_page(host[i], n, float(eb), idx, src, epl)
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want)


# 4112 tiles: two per workgroup, up to 16 shards a job; 8198: four and 32.
# Whole blocks run on the persistent encoder for long jobs, cut ones do not.
@pytest.mark.parametrize("count,n,off", [(16, LONG + 8192, 0), (16, LONG + 4096 + 17, 1),
                                         (2, 4099 * 8192, 0)])
def test_several_tiles_per_workgroup(oracle, count, n, off):
    pages = flat_pages(count, n, off, torch.bfloat16, count)
    for i in range(count):   # each job's own extremes, next to its neighbours'
        pages[i, 0], pages[i, -1] = 10.0 + i, -20.0 - 3 * i
    w = fixed_wrapper()
    bufs = [buffer(n) for _ in range(count)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16(list(pages), bufs, [1e-4] * count)
    assert ok
    host = bits(pages)
    want, _, want_bounds = oracle.compress_batch(host, [1e-4] * count, relative=True, threads=8)
    for i in range(count):
        assert np.float32(bounds[i]) == np.float32(want_bounds[i]), i
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want[i]), i


@pytest.mark.parametrize("mode", ["fixed", "plain", "outlier"])
@pytest.mark.parametrize("n,off", [(LONG + 2048 + 33, 3), (LONG + 2047, 0), (300 * 8192, 1)])
def test_long_fp32_pages(oracle, mode, n, off):
    import cuszp_wrapper_cpp as cpp

    m = {"fixed": cpp.MODE_FIXED, "plain": cpp.MODE_PLAIN, "outlier": cpp.MODE_OUTLIER}[mode]
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(1e-4, True, cpp.DIM_1D, m, cpp.TYPE_FLOAT), 0)
    kinds = 6
    pages = flat_pages(kinds, n, off, torch.float32, n)
    pages[0, 0], pages[0, -1] = -9.0, 7.0
    pages[1] = pages[1].abs() + 0.5
    pages[2] = -pages[2].abs()
    pages[2, -1] = -60.0
    pages[3] = 0.0
    pages[3, -1] = -0.0
    pages[4, -1] = float("nan")
    pages[5, 0], pages[5, -1] = float("inf"), -3.0
    host = pages.cpu().numpy()
    for i in range(kinds):
        buf = torch.full((8 * n + 1024 + 136,), 0xAB, dtype=torch.uint8, device="cuda")
        ok, buf, size, bound = w.compress(pages[i], buf, 1e-4)
        assert ok
        eb = np.float32(oracle.relative_bound_f32(host[i], 1e-4))
        assert np.float32(bound) == eb or (np.isnan(eb) and np.isnan(bound)), i
        want = (oracle.compress_page_f32(host[i], float(eb)) if mode == "fixed"
                else oracle.compress_page_f32_mode(host[i], float(eb), int(m)))
        assert size == want.size, i
        assert np.array_equal(buf[:size].cpu().numpy(), want), i
        assert bool((buf[size:] == 0xAB).all()), i


@pytest.mark.parametrize("n", [1, 31, 2047, 2048, 8193, 5 * 8192 + 33])
def test_fp32_pages(oracle, n):
    kinds = 6
    pages = flat_pages(kinds, n, 3, torch.float32, n)
    pages[0, -1] = 7.0
    pages[1] = pages[1].abs()
    pages[2] = -pages[2].abs()
    pages[3] = 0.0
    pages[3, -1] = -0.0
    pages[4, n // 2] = float("nan")
    pages[5, 0], pages[5, -1] = float("inf"), -3.0
    w = fixed_wrapper()
    bufs = [buffer(n) for _ in range(kinds)]
    ok, sizes, bounds = w.compress_batch_fixed(list(pages), bufs, [1e-4] * kinds)
    assert ok
    host = pages.cpu().numpy()
    for i in range(kinds):
        eb = np.float32(oracle.relative_bound_f32(host[i], 1e-4))
        assert np.float32(bounds[i]) == eb or (np.isnan(eb) and np.isnan(bounds[i]))
        want = oracle.compress_page_f32(host[i], float(eb))
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want)
