"""What a warm-ahead hint points into is held as long as a launch may read it.  rtp_gemm_warm_next keeps one hint: a later call
ends it, also one from another thread, because only the memory of the last hint is held (a backward pass rotates on the
autograd engine's thread).  A hint that a capture recorded is read at every replay."""
import gc
import os
import threading
import weakref

import pytest
import torch

from rtp_amd import _lib, emulate_shards, ring
from rtp_amd.module.linear import ColumnParallelLinear


def _in_thread(fn):
    got = []
    t = threading.Thread(target=lambda: got.append(fn()))
    t.start()
    t.join()
    return got[0]


@pytest.mark.parametrize("later", [True, False])
def test_another_threads_call_ends_a_pending_hint(later):
    lib = _lib.load()
    a, b = torch.zeros(64), torch.zeros(64)
    assert lib.rtp_gemm_warm_next(a.data_ptr(), 256) == 0 and lib.rtp_gemm_warm_pending() == 1
    assert _in_thread(lib.rtp_gemm_warm_pending) == 0          # a hint is its own thread's

    def other():
        src, size = (b.data_ptr(), 256) if later else (None, 0)
        lib.rtp_gemm_warm_next(src, size)
        return lib.rtp_gemm_warm_pending()

    assert _in_thread(other) == int(later)
    assert lib.rtp_gemm_warm_pending() == 0
    assert lib.rtp_gemm_warm_next(a.data_ptr(), 256) == 0 and lib.rtp_gemm_warm_pending() == 1
    assert lib.rtp_gemm_warm_next(None, 0) == 0 and lib.rtp_gemm_warm_pending() == 0


@pytest.mark.skipif(not os.path.exists(_lib.NATIVE_PATH), reason="_rtp_native.so not built")
@pytest.mark.parametrize("window", [None, 1])
def test_rows_that_a_captured_launch_reads_live_as_long_as_its_layer(monkeypatch, window):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)  # hints are only set for device tensors; nothing is launched here
    capturing = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capturing))
    was = ring.warm_ahead()
    ring.set_warm_ahead(True)  # forgets what was learned
    ring.set_rotation_window(window)
    try:
        with emulate_shards(2):
            mine, other, third = (ColumnParallelLinear(8, 4) for _ in range(3))
        for layer in (mine, other, third, mine, other, third):  # three programs in turn: other follows mine
            ring.rotation(layer._store, 0)
        assert not any(layer._store.captured_hints for layer in (mine, other, third))
        capturing.append(True)
        ring.rotation(mine._store, 0)
        capturing.clear()
        rows = weakref.ref(other._store.home)
        assert mine._store.captured_hints[rows().data_ptr()] is rows()
        del other, layer
        ring.rotation(third._store, 0)  # the pending hint is replaced
        ring.set_warm_ahead(True)
        gc.collect()
        assert rows() is not None       # a replay would read it
        del mine
        gc.collect()
        assert rows() is None
    finally:
        ring.set_rotation_window(None)
        ring.set_warm_ahead(was)
