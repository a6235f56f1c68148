"""A recorded step() reads its chunk table by address at every replay: the table lives as long as its optimiser, whatever later
steps and captures leave to be updated.  On the CPU, with the launches left out."""
import gc
import weakref

import pytest
import torch

from rtp_amd import emulate_shards, ops, optim, ring
from rtp_amd.module.linear import ColumnParallelLinear


@pytest.fixture
def world(monkeypatch):
    """What a step launched, as weak references to the tables; `capturing` is true while it is not empty."""
    launched, capturing = [], []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capturing))
    monkeypatch.setattr(ring, "join_wgrad", lambda *a: None)
    monkeypatch.setattr(ring, "fence", lambda *a: None)
    monkeypatch.setattr(ops, "sgd_step", lambda *a: launched.append(None))
    monkeypatch.setattr(ops, "adam_step", lambda *a: launched.append(None))
    monkeypatch.setattr(ops, "sgd_step_multi", lambda table, *a: launched.append(weakref.ref(table)))
    monkeypatch.setattr(ops, "adam_step_multi", lambda table, *a: launched.append(weakref.ref(table)))
    return launched, capturing


def _model(n_out, dtype=torch.float32):
    with emulate_shards(2):
        layers = [ColumnParallelLinear(8, n_out, dtype=dtype) for _ in range(2)]
    for layer in layers:
        layer._store.grads = torch.zeros_like(layer._store.home)
    return torch.nn.ModuleList(layers), [layer._store for layer in layers]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n_out", [6, 16])  # slices of 24 and 3 elements, and of 64 and 8
@pytest.mark.parametrize("later", ["eager", "capture"])
def test_table_of_a_fused_step(world, dtype, n_out, later):
    launched, capturing = world
    model, stores = _model(n_out, dtype)
    opt = optim.RotatedSGD(model, 0.1, fused_backward=True)

    def step(products):
        for st in products:  # whose weight-gradient products have updated the weights
            st.fused_sgd.applied = {(st.offsets[0], st.numels[0]): {0, 1}}
        opt.step()

    step(stores)
    capturing.append(True)
    step(stores)
    recorded = launched[-1]
    assert recorded is not None and recorded() is not None
    if later == "capture" and n_out == 16:
        with pytest.raises(RuntimeError):  # an aligned table cannot be made under capture
            step(stores[:1])
    elif later == "capture":
        step(stores[:1])                   # odd slices: launched one by one
        assert launched[-1] is None
    else:
        capturing.clear()
        step(stores[:1])                   # a step in which one layer takes no part
    capturing.clear()
    step(stores)
    gc.collect()
    assert recorded() is not None
    del opt
    for st in stores:
        st.fused_sgd = None
    gc.collect()
    assert recorded() is None


@pytest.mark.parametrize("adam", [False, True])
def test_table_of_a_step_over_all_buffers(world, adam):
    launched, capturing = world
    model, stores = _model(6)
    opt = optim.RotatedAdam(model) if adam else optim.RotatedSGD(model, 0.1)
    opt.step()
    capturing.append(True)
    opt.step()
    recorded = launched[-1]
    assert recorded is not None
    capturing.clear()
    if adam:
        stores[1].grads = None             # a layer that has no gradients yet
    else:
        stores[1].grads = stores[1].grads.clone()
    opt.step()
    gc.collect()
    assert launched[-1] is not recorded and recorded() is not None
