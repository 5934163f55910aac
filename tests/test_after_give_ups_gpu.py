"""Calls after persistent encoder launches that gave up: three in a row send the
context's next 64 calls of at least as many tiles to one workgroup per tile,
smaller calls and contexts with KVSZP_SAFE_CALLS keep trying.  Give-ups are forced
with a wait bound of zero.  Streams and bounds against the oracle throughout."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import fixed_wrapper

pytestmark = pytest.mark.gpu

ROW, AFTER = 3, 64

# (pages, values of each, offset): thousands of tiles, so that some wait of a
# launch is not met at its first poll: long jobs, whole blocks at an odd
# address, segments that end inside a block
CALLS = [(2, 4096 * 8192, 0), (300, 28 * 8192, 1), (300, 28 * 8192 - 5, 0)]


class Store:
    def __init__(self, oracle, w, count, n, off, entry="wrapper"):
        g = torch.Generator().manual_seed(n)
        flat = torch.randn(off + count * n, generator=g).to(torch.bfloat16).cuda()
        self.pages = flat[off:].view(count, n)
        self.w, self.entry, self.n = w, entry, n
        host = self.pages.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)
        self.want, _, self.bounds = oracle.compress_batch(host, [1e-4] * count, relative=True,
                                                          threads=8)
        self.bufs = [torch.empty(8 * n, dtype=torch.uint8, device="cuda") for _ in range(count)]

    def __call__(self, check=True):
        count = len(self.bufs)
        if check:
            for b in self.bufs:
                b.fill_(0xAB)
        if self.entry == "wrapper":
            ok, sizes, bounds = self.w.compress_batch_fixed_bf16(list(self.pages), self.bufs,
                                                                 [1e-4] * count)
            assert ok
        else:
            import kvszp

            sizes, bounds = (ctypes.c_uint64 * count)(), (ctypes.c_float * count)()
            kvszp.check(self.w._ctx.compress_noalloc(
                kvszp.ptr_array([p.data_ptr() for p in self.pages]),
                kvszp.ptr_array([b.data_ptr() for b in self.bufs]),
                kvszp.u64_array([8 * self.n] * count), None, count, self.n,
                torch.cuda.current_stream().cuda_stream, sizes, bounds))
        if check:
            for i in range(count):
                assert np.float32(bounds[i]) == np.float32(self.bounds[i]), i
                assert sizes[i] == self.want[i].size, i
                assert np.array_equal(self.bufs[i][:sizes[i]].cpu().numpy(), self.want[i]), i


@pytest.mark.parametrize("entry", ["wrapper", "no allocation"])
@pytest.mark.parametrize("count,n,off", CALLS)
def test_three_in_a_row(oracle, count, n, off, entry):
    w = fixed_wrapper()
    counts = w._ctx.schedule_counts
    store = Store(oracle, w, count, n, off, entry)
    small = Store(oracle, w, 5, 9 * 8192, 0, entry)
    w._ctx.set_wait_bound(0)
    for _ in range(20):
        store()
        if counts()["safe_calls"]:
            break
    w._ctx.set_wait_bound(200)
    tried = counts()["reencoded"]
    assert tried >= ROW and counts()["safe_calls"] == 1
    store()
    small()                                     # not counted, and on the persistent encoder
    assert counts()["safe_calls"] == 2
    for _ in range(AFTER - 2):
        store(check=False)
    assert counts()["safe_calls"] == AFTER
    store()                                     # tries again
    assert counts()["safe_calls"] == AFTER


def test_explicit_setting_turns_it_off(oracle, monkeypatch):
    monkeypatch.setenv("KVSZP_SAFE_CALLS", "0")
    w = fixed_wrapper()
    w._ctx.set_wait_bound(0)
    store = Store(oracle, w, *CALLS[1])
    for _ in range(2 * ROW):
        store()
    assert w._ctx.schedule_counts()["safe_calls"] == 0
    assert w._ctx.reencode_count() >= ROW
