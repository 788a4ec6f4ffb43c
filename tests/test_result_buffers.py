"""The page-locked buffers behind an engine's logits arrays: used again only when every view of the array is gone,
bounded, given back at close and after it, and replaced by ordinary arrays past the bound or without the memory.
No GPU: the two C calls are replaced by a counted heap."""
import ctypes as C
import threading

import numpy as np
import pytest

from retrograd_amd.engine import _ResultBuffers


class _Heap:
    def __init__(self, refuse=False):
        self.live, self.refuse, self.made = {}, refuse, 0

    def retro_host_alloc(self, n):
        if self.refuse:
            return None
        block = C.create_string_buffer(n)
        self.live[C.addressof(block)] = block
        self.made += 1
        return C.addressof(block)

    def retro_host_free(self, at):
        del self.live[at]


MB = 1 << 18          # floats of one megabyte


@pytest.mark.parametrize("shape", [(4, MB), (1, MB), (3, MB + 7)])
def test_a_buffer_comes_back_when_the_last_view_is_gone(shape):
    heap = _Heap()
    pool = _ResultBuffers(heap)
    a = pool.take(shape)
    assert a.shape == shape and a.dtype == np.float32 and a.flags.c_contiguous and a.flags.writeable
    a[:] = 3.0
    tail, at = a[-1, -5:], a.ctypes.data
    del a
    b = pool.take(shape)                       # the view keeps the first buffer
    assert b.ctypes.data != at
    b[:] = 4.0
    assert (tail == 3.0).all()
    del tail
    assert pool.take(shape).ctypes.data == at and heap.made == 2


def test_small_results_and_refused_memory_are_ordinary_arrays():
    heap = _Heap()
    assert _ResultBuffers(heap).take((1, MB - 1)).flags.owndata and not heap.live
    assert _ResultBuffers(heap).take((0, MB)).shape == (0, MB)
    assert _ResultBuffers(_Heap(refuse=True)).take((4, MB)).flags.owndata


def test_the_bound_holds_for_kept_results_and_for_changing_sizes():
    heap = _Heap()
    pool = _ResultBuffers(heap)
    kept = [pool.take((32, MB)) for _ in range(6)]
    assert [a.flags.owndata for a in kept] == [False] * 4 + [True] * 2 and len(heap.live) == 4
    kept.clear()
    for n in (1, 5, 17, 40, 100, 128, 3, 129):
        a = pool.take((n, MB))
        assert a.shape == (n, MB) and sum(len(b) for b in heap.live.values()) <= pool.LIMIT_BYTES
    assert a.flags.owndata                     # larger than the bound


def test_close_frees_what_waits_and_live_arrays_free_their_own_on_any_thread():
    heap = _Heap()
    pool = _ResultBuffers(heap)
    box = [pool.take((8, MB)), pool.take((8, MB))]
    box[0][:] = 1.0
    del box[1]
    pool.close()
    assert len(heap.live) == 1 and (box[0] == 1.0).all()
    t = threading.Thread(target=box.clear)
    t.start()
    t.join()
    assert not heap.live
    assert pool.take((8, MB)).flags.owndata
