"""The library's own reuse of freed device blocks: statistics count them as free, they go back on request and above the
release threshold, results stay right while blocks are handed out again under queued work and from several threads."""
import threading

import numpy as np
import pytest

import ctorch_amd as ct
from common import say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


def full(n, value):
    return ct.Tensor(ct._new(ct.lib().dl_full, ct._shape([n]), value, ct.options()))


def test_freed_blocks_count_as_free_and_go_back_on_request():
    say("case: block reuse statistics, release and threshold")
    ct.release_unused()
    before = ct.memory_stats()
    held = [full(1 << 18, 1.0) for _ in range(8)]
    live = ct.memory_stats()
    assert live.used_bytes - before.used_bytes == 8 << 20
    del held
    freed = ct.memory_stats()
    assert freed.used_bytes == before.used_bytes and freed.peak_used_bytes >= live.used_bytes
    again = [full(1 << 18, 2.0) for _ in range(8)]  # the same blocks
    assert ct.memory_stats().reserved_bytes == freed.reserved_bytes
    assert all(np.all(t.numpy() == 2.0) for t in again)
    del again
    ct.release_unused()
    assert ct.memory_stats().reserved_bytes <= before.reserved_bytes
    keep = ct.memory_stats().release_threshold
    try:
        ct.set_release_threshold(0)
        held = [full(1 << 20, 3.0) for _ in range(32)]
        with_them = ct.memory_stats().reserved_bytes
        del held  # to the runtime, whose pool gives up what it has above the threshold when the stream is waited for
        ct.synchronize()
        freed = ct.memory_stats()
        say(f"  reserved {before.reserved_bytes} -> {with_them} -> {freed.reserved_bytes}")
        assert freed.used_bytes == before.used_bytes and freed.reserved_bytes <= with_them - (64 << 20)
    finally:
        ct.set_release_threshold(keep)


def test_blocks_are_reused_in_order_from_several_threads():
    say("case: four threads allocate, compute on and free blocks of the same sizes")
    rng = np.random.default_rng(0)
    x = rng.standard_normal((4, 8, 64)).astype(np.float32)
    w = rng.standard_normal((96, 64)).astype(np.float32)
    gw = ct.Tensor.from_numpy(w, ct.F32, GPU)
    wrong = []

    def work(i):
        gx = ct.Tensor.from_numpy(x[i], ct.F32, GPU)
        want = ct.linear(gx, gw).numpy()
        for _ in range(200):
            y = ct.linear(gx, gw)
            z = ct.linear(gx, gw)
            del y  # its block may be the next result's while the launch that wrote it is still queued
            y = ct.linear(gx, gw)
            if not (np.array_equal(z.numpy(), want) and np.array_equal(y.numpy(), want)):
                wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
