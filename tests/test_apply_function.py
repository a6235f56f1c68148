"""apply_function: a function's forward alone where gradients are off and nothing else takes hold of it; its apply everywhere else."""
import pytest
import torch
from torch.autograd import forward_ad

from rtp_amd.module.utils import apply_function


class _Twice(torch.autograd.Function):
    calls = []

    @staticmethod
    def forward(ctx, x, other=None):
        _Twice.calls.append(type(ctx).__name__)
        ctx.save_for_backward(x)
        ctx.note = other
        y = torch.empty(x.numel(), dtype=x.dtype)
        y.copy_(2 * x.reshape(-1))
        return y.view(*x.shape[:-1], x.shape[-1])

    @staticmethod
    def backward(ctx, dy):
        return 2 * dy, None


def _plain():
    return _Twice.calls.pop() == "_NoGradContext"


def test_without_gradients_the_forward_runs_alone():
    x = torch.randn(2, 3, 4, requires_grad=True)
    with torch.no_grad():
        y = apply_function(_Twice, x)
    assert _plain() and y.grad_fn is None and not y.requires_grad and torch.equal(y, 2 * x.detach())
    with torch.inference_mode():
        y = apply_function(_Twice, x, 3)
    assert _plain() and y.is_inference()


def test_with_gradients_it_is_apply():
    x = torch.randn(2, 3, requires_grad=True)
    apply_function(_Twice, x).sum().backward()
    assert not _plain() and torch.equal(x.grad, torch.full((2, 3), 2.0))


def test_forward_mode_is_refused_as_by_apply():
    x = torch.randn(2, 3)
    with torch.no_grad(), forward_ad.dual_level():
        d = forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(RuntimeError):
            _Twice.apply(d)
        with pytest.raises(RuntimeError):
            apply_function(_Twice, d)
    _Twice.calls.clear()


def test_transforms_are_refused_as_by_apply():
    for f in (lambda x: _Twice.apply(x), lambda x: apply_function(_Twice, x)):
        with torch.no_grad(), pytest.raises(RuntimeError):
            torch.func.vmap(f)(torch.randn(2, 3))
    assert not _Twice.calls


def test_a_tracer_sees_apply():
    with torch.no_grad():
        torch.jit.trace(lambda x: apply_function(_Twice, x), torch.randn(2, 3), check_trace=False)
    assert _Twice.calls and "_NoGradContext" not in _Twice.calls
    _Twice.calls.clear()


def test_results_of_either_refuse_a_later_in_place_use_alike():
    """A view made inside the function, changed in place by something that wants gradients."""
    p = torch.randn(2, 3, requires_grad=True)
    for f in (lambda x: _Twice.apply(x), lambda x: apply_function(_Twice, x)):
        with torch.no_grad():
            y = f(torch.randn(2, 3))
        with pytest.raises(RuntimeError):
            y += p
    _Twice.calls.clear()


@pytest.mark.parametrize("where,name", [(torch._C, "_are_functorch_transforms_active"), (torch._C, "_get_tracing_state"),
                                        (torch._C._functorch, "unwrap_if_dead"), (forward_ad, "_current_level")])
def test_in_a_torch_without_one_of_the_names_it_is_apply(where, name, monkeypatch):
    import importlib.util

    import rtp_amd.module.utils as utils
    with monkeypatch.context() as m:
        m.delattr(where, name)
        spec = importlib.util.spec_from_file_location("utils_of_another_torch", utils.__file__)
        other = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(other)
    with torch.no_grad():
        other.apply_function(_Twice, torch.randn(2, 3))
    assert not _plain()


def test_a_subclass_with_a_function_of_its_own():
    """It may use all of apply's context, and hand an argument back."""
    from rtp_amd import emulate_shards
    from rtp_amd.module.linear import ColumnParallelLinear

    class Own(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, anchor, layer):
            ctx.set_materialize_grads(False)
            assert ctx.needs_input_grad[0] == x.requires_grad
            ctx.mark_dirty(x)
            return x.add_(1)

    class Layer(ColumnParallelLinear):
        _fn = Own

    with emulate_shards(2):
        layer = Layer(8, 4)
    x = torch.zeros(3, 8)
    for off in (torch.no_grad, torch.inference_mode):
        with off():
            assert layer(x) is x
    assert torch.equal(x, torch.full((3, 8), 2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layers_give_the_same_with_and_without_gradients(dtype):
    from rtp_amd import emulate_shards
    from rtp_amd.models.transformer_lm_rtp import TransformerLM
    from rtp_amd.module.conv import ColumnParallelConv2d
    from rtp_amd.module.linear import ColumnParallelLinear, RowParallelLinear
    dev = "cuda:0"
    torch.manual_seed(1)
    with emulate_shards(2):
        layers = [(ColumnParallelLinear(64, 96, device=dev, dtype=dtype), (5, 3, 64)),
                  (RowParallelLinear(64, 40, device=dev, dtype=dtype), (7, 64)),
                  (ColumnParallelConv2d(3, 8, 3, device=dev, dtype=dtype), (2, 3, 9, 9))]
    lm = TransformerLM(96, 64, 2, 64, 0.0, 0.1, 2, 2, 0, device=dev, dtype=dtype)
    cases = [(layer, torch.randn(*shape, device=dev, dtype=dtype)) for layer, shape in layers]
    cases.append((lm, torch.randint(0, 96, (8, 2), device=dev)))
    for layer, x in cases:
        with_grad = layer(x)
        with torch.no_grad():
            without = layer(x)
        assert with_grad.requires_grad and not without.requires_grad
        assert torch.equal(with_grad.detach(), without)
