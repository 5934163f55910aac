"""The persistent encoder on segments that end inside a block and pages at any
2-byte address: the cut block in either wave and either half of a tile, alone
in a tile, holding the extremes, a NaN or one value; bounds that overflow the
staging, or whose reciprocal is infinite or negative.  Streams, sizes and
bounds against the oracle, through both entry points."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def pages_of(n, off):
    g = torch.Generator().manual_seed(n)
    x = torch.randn(7, n, generator=g)
    x[1, -1], x[2, -1] = 40.0, -40.0            # an extreme in the cut block
    x[3] = 1.3125                               # one value: rates up to 31
    x[4] = 0.0
    x[4, -1] = 2.0
    x[5, -1] = float("nan")
    x[6] = x[6].abs() + 0.25                    # zeros would widen the range
    flat = torch.zeros(off + x.numel(), dtype=torch.bfloat16, device="cuda")
    flat[off:] = x.to(torch.bfloat16).flatten().cuda()
    return flat[off:].view(7, n)


def check(oracle, pages, n, eps, relative, bufs, sizes, bounds):
    host = bits(pages)
    for i in range(len(bufs)):
        eb = np.float32(oracle.relative_bound(host[i], n, eps) if relative else eps)
        assert np.float32(bounds[i]) == eb, i
        want = oracle.compress_page(host[i], n, float(eb))
        assert sizes[i] == len(want), (i, sizes[i], len(want))
        assert np.array_equal(bufs[i][:sizes[i]].cpu().numpy(), want), i
        assert bool((bufs[i][sizes[i]:] == 0xAB).all()), i


# bound: relative, absolute, absolute with an infinite reciprocal, negative
# (-0.0: its reciprocal is -inf)
@pytest.mark.parametrize("eps,relative", [(1e-4, True), (1e-3, False), (1e-40, False),
                                          (-1e-2, False), (-1e-4, True), (-0.0, False),
                                          (-0.0, True)])
@pytest.mark.parametrize("n,off", [(1, 1), (31, 0), (33, 3), (2047, 1), (2049, 0), (4095, 5),
                                   (4097, 1), (6145, 0), (8191, 7), (8193, 1),
                                   (5 * 8192 + 4096, 0), (5 * 8192 + 4096, 1), (30 * 8192 + 2080 + 17, 3)])
def test_cut_blocks(oracle, n, off, eps, relative):
    import cuszp_wrapper_cpp as cpp

    pages = pages_of(n, off)
    w = cpp.CuSZpWrapper(cpp.CompressionConfig(eps, relative, cpp.DIM_1D, cpp.MODE_FIXED,
                                               cpp.TYPE_FLOAT), 0)
    cap = max(8 * n, 1024 * -(-n // 32768) + 128 * -(-n // 32))
    bufs = [torch.full((cap,), 0xAB, dtype=torch.uint8, device="cuda") for _ in range(7)]
    ok, sizes, bounds = w.compress_batch_fixed_bf16(list(pages), bufs, [])
    assert ok
    check(oracle, pages, n, eps, relative, bufs, sizes, bounds)


@pytest.mark.parametrize("n,off", [(33, 1), (4097, 0), (3 * 8192 + 95, 3)])
def test_cut_blocks_no_allocation(oracle, n, off):
    import ctypes

    import kvszp

    pages = pages_of(n, off)
    cap = max(8 * n, 1024 * -(-n // 32768) + 128 * -(-n // 32))
    bufs = [torch.full((cap,), 0xAB, dtype=torch.uint8, device="cuda") for _ in range(7)]
    ctx = kvszp.Context(kvszp.Config(1e-4, 1, kvszp.DIM_1D, kvszp.MODE_FIXED,
                                     kvszp.TYPE_FLOAT), 0)
    sizes, bounds = (ctypes.c_uint64 * 7)(), (ctypes.c_float * 7)()
    kvszp.check(ctx.compress_noalloc(
        kvszp.ptr_array([p.data_ptr() for p in pages]),
        kvszp.ptr_array([b.data_ptr() for b in bufs]), kvszp.u64_array([cap] * 7), None, 7, n,
        torch.cuda.current_stream().cuda_stream, sizes, bounds))
    check(oracle, pages, n, 1e-4, True, bufs, list(sizes), list(bounds))
