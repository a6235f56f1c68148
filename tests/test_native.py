"""The extension module of csrc/host.cpp on the CPU: attaching gradient slices (GradBook) and argument errors.  Its product
and kernel calls are what every GPU test runs through."""
import os

import pytest
import torch

from rtp_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.NATIVE_PATH), reason="_rtp_native.so not built")


def _layer():
    params = [[torch.nn.Parameter(torch.zeros(2, 3)), torch.nn.Parameter(torch.zeros(3))] for _ in range(2)]
    grads = torch.arange(18.0).view(2, 9)
    views = [[row[:6].view(2, 3), row[6:]] for row in grads]
    return params, grads, views, _lib.native().GradBook(params, views)


def test_grad_book_attaches_accumulates_and_leaves_mixed_states_alone():
    params, grads, views, book = _layer()
    assert book.attach() == 0 and not grads.equal(torch.zeros_like(grads))      # attached, contents left to the kernels
    for ps, vs in zip(params, views):
        for p, v in zip(ps, vs):
            assert p.grad.data_ptr() == v.data_ptr() and p.grad.shape == p.shape
    assert book.complete() and book.attach() == 1                               # every slice in place: accumulate
    params[1][0].grad = None
    assert not book.complete() and book.attach() == -1                          # one shard fresh, one not
    assert params[1][0].grad is None
    params[1][0].grad = torch.ones(2, 3)
    assert book.complete() and book.attach() == -1                              # somebody's own tensor
    book.drop()
    assert all(p.grad is None for ps in params for p in ps)
    params[0][1].grad = params[1][1].grad = torch.ones(3)
    assert book.attach() == 0                                                   # some parameter of every shard is fresh
    assert params[0][1].grad.data_ptr() == views[0][1].data_ptr()


def test_argument_errors():
    n = _lib.native()
    with pytest.raises(ValueError):
        n.GradBook([[torch.zeros(1)]], [[]])
    with pytest.raises(TypeError):
        n.gemm(torch.float16, m=1)
    with pytest.raises(TypeError):
        n.gemm(torch.float32, rows=1)
    with pytest.raises(TypeError):
        n.rtp_layernorm_supported(0)
    with pytest.raises(_lib.RtpError):
        n.linear_fwd(torch.zeros(2, 4), torch.zeros(1, 8), 0, None, 2, 4, torch.zeros(2, 2), 0, False)
    assert n.rtp_attn_supported(_lib.RTP_BF16, 32, 64) == 1 and n.rtp_attn_supported(_lib.RTP_F32, 32, 64) == 0


def test_a_tensor_without_plain_storage_raises():
    """data_ptr(), strides and sizes throw in C++ for such tensors; every function turns that into a Python error."""
    n = _lib.native()
    sparse = torch.eye(4).to_sparse()
    with pytest.raises(RuntimeError):
        n.gemm(torch.float32, a=sparse, m=1)
    with pytest.raises(RuntimeError):
        n.rtp_gemm_warm_next(sparse, 0)
    with pytest.raises((RuntimeError, ValueError)):
        n.linear_fwd(torch.zeros(2, 4), sparse, 0, None, 2, 4, torch.zeros(2, 2), 0, False)
    with pytest.raises((RuntimeError, ValueError)):
        n.linear_bwd(sparse, 0, None, sparse, 0, None, 1, 4, None, None, None, None, False, None, None, 0.0, 0.0, False)
    seen = []

    def probe(x):  # a functorch tensor has no storage of its own
        with pytest.raises(RuntimeError):
            n.rtp_gemm_warm_next(x, 0)
        seen.append(x)
        return x.sum()

    torch.func.grad(probe)(torch.ones(3))
    assert len(seen) == 1


def test_grad_book_with_a_gradient_of_another_layout():
    params, grads, views, book = _layer()
    book.attach()
    w, b = params[0]
    w.grad = torch.ones(2, 3).to_sparse()
    with pytest.raises(RuntimeError):
        book.attach()
    assert w.grad.is_sparse and book.complete()                                 # nothing was attached
    b.grad = None                                                               # a fresh shard is attached as a whole
    params[1][0].grad = None
    assert book.attach() == 0 and w.grad.data_ptr() == views[0][0].data_ptr()
    w.grad = torch.ones(2, 3).to_sparse()
    book.drop()
    assert w.grad is None
