"""rtp_gemm_warm_next keeps one hint: a later call ends it, also one from another thread, because only the memory of the last
hint is held (a backward pass rotates on the autograd engine's thread)."""
import threading

import pytest
import torch

from rtp_amd import _lib


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
