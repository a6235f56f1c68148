"""Copies of a rotated layer (copy.deepcopy, pickle, torch.save) before and after its first backward: values, the parameters'
place in the copy's flat buffers, nothing shared with the original, and the gradient state a backward finds there."""
import copy
import io
import os
import pickle

import pytest
import torch
import torch.nn as nn

from rtp_amd import _lib, emulate_shards
from rtp_amd.module import attention, linear

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.NATIVE_PATH), reason="_rtp_native.so not built")


def _through_file(layer):
    f = io.BytesIO()
    torch.save(layer, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


def _column():
    with emulate_shards(4):
        return linear.ColumnParallelLinear(12, 8)


def _attention():
    return attention.ParallelMultiheadAttention(8, 4, 2, 0, MultiheadAttention_layer=nn.MultiheadAttention(8, 4))


@pytest.mark.parametrize("make", [_column, _attention])
@pytest.mark.parametrize("how", [copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m)), _through_file],
                         ids=["deepcopy", "pickle", "torch.save"])
@pytest.mark.parametrize("after_backward", [False, True])
def test_copies_keep_the_flat_storage(make, how, after_backward):
    layer = make()
    store = layer._store
    ws = store.world_size
    if after_backward:
        assert store.grad_runs() == [(0, ws, False)]
        store.grads.fill_(3.0)
    other = how(layer)
    mine = other._store
    assert mine.home.equal(store.home) and mine.home.data_ptr() != store.home.data_ptr()
    assert mine.one_run.acquire(0)[0][0] is mine.home
    for s, sub in enumerate(mine.modules):
        assert sub is other.shards[s] and sub._full_param.data_ptr() == mine.home[s].data_ptr()
        for p, v in zip(sub.parameters(), mine.views(mine.home[s])):
            assert p.data_ptr() == v.data_ptr() and p.shape == v.shape and p.grad is None
    with torch.no_grad():
        next(other.parameters()).add_(1.0)
    assert not mine.home.equal(store.home)
    # the copy's parameters carry no gradients: its first backward overwrites, its second accumulates
    assert mine.grad_runs() == [(0, ws, False)] and mine.grad_runs() == [(0, ws, True)]
    for s, sub in enumerate(mine.modules):
        assert sub._full_grad.data_ptr() == mine.grads[s].data_ptr()
        for p, v in zip(sub.parameters(), mine.views(mine.grads[s])):
            assert p.grad.data_ptr() == v.data_ptr()
    if after_backward:  # the original goes on as if nothing had happened
        assert mine.grads.data_ptr() != store.grads.data_ptr() and store.grad_runs() == [(0, ws, True)]
        other.zero_grad()
        assert all(p.grad is None for p in other.parameters()) and all(p.grad is not None for p in layer.parameters())


def test_gradients_put_on_a_copy_are_accumulated_into():
    layer = _column()
    layer._store.grad_runs()
    other = copy.deepcopy(layer)
    for p in other.parameters():
        p.grad = torch.full_like(p, 2.0)
    assert other._store.grad_runs() == [(0, 4, True)]
    assert all(v.eq(2.0).all() for s in range(4) for v in other._store.views(other._store.grads[s]))


def test_zero_grad_with_an_empty_child_slot():
    layer = _column()
    layer._store.grad_runs()
    layer.register_module("extra", None)  # as torch modules may have
    layer.zero_grad()
    assert all(p.grad is None for p in layer.parameters())
