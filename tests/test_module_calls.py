"""What a program may do to the quantized layers' calls from Python, whatever the native path does: trace and replace them."""
import pytest
import torch
import torch.nn.functional as F

from khaosz_amd import QuantLinear


def _float_forward(self, x, residual=None, norm=None):
    y = F.linear(x, self.qweight.to(x.dtype)) * self.w_scale
    return y if residual is None else y + residual


class _Float(QuantLinear):
    """The layer in torch's own operators, for a machine without the GPU."""
    forward = _float_forward


def _layer(cls):
    q = cls(32, 16)
    q.qweight.random_(-100, 100, generator=torch.Generator().manual_seed(1))
    return q, torch.randn(4, 32, generator=torch.Generator().manual_seed(2))


@pytest.fixture(params=[False, True], ids=["before", "after"])
def told(request):
    """Before and after the process's first call of a layer that goes to native code."""
    from khaosz_amd import linear
    if request.param:
        linear.linear_native()
    return request.param


@pytest.mark.parametrize("inside", [False, True])
def test_a_subclass_with_a_forward_of_its_own_compiles_without_a_graph_break(told, inside):
    q, x = _layer(_Float)
    want = q(x)
    torch._dynamo.reset()
    f = torch.compile((lambda x: q(x) * 2) if inside else q, fullgraph=True, backend="eager")
    assert torch.equal(f(x), want * 2 if inside else want)
    h = q.register_forward_hook(lambda m, a, y: y * 2)
    assert torch.equal(torch.compile(lambda x: q(x), fullgraph=True, backend="eager")(x), want * 2)
    h.remove()


def test_a_subclass_is_traced_by_fx_and_export(told):
    q, x = _layer(_Float)
    model = torch.nn.Sequential(q, torch.nn.ReLU())
    assert torch.equal(torch.fx.symbolic_trace(model)(x), model(x))
    assert torch.equal(torch.export.export(model, (x,)).module()(x), model(x))


def test_a_forward_replaced_on_the_class_is_compiled_without_a_graph_break(monkeypatch, told):
    q, x = _layer(QuantLinear)
    monkeypatch.setattr(QuantLinear, "forward", _float_forward)
    want = _float_forward(q, x)
    torch._dynamo.reset()
    assert torch.equal(q(x), want) and torch.equal(torch.compile(q, fullgraph=True, backend="eager")(x), want)


def test_the_native_rule_for_the_merge_inside_the_projection_is_the_operators():
    from khaosz_amd import block, ops
    block._native()
    host = ops._native()
    for B in range(0, 12):
        for heads, d in ((1, 64), (8, 64), (24, 64), (31, 64), (32, 64), (16, 128), (17, 128), (33, 64)):
            for total in (1, 255, 256, 257, 512, 513, 768, 769, 1024, 1025, 5000):
                assert host.attn_gemv_fusable(B, heads * d, total) == ops.attn_gemv_fusable(B, heads, d, total)


def test_what_native_code_leaves_goes_to_the_next_call_behind_the_layers(monkeypatch, told):
    """As the Python code of their ``__call__`` would have it: a base class's call, or nn.Module's as it is now."""
    seen = []

    class Watched(torch.nn.Module):
        def __call__(self, *args, **kwargs):
            seen.append(kwargs)
            return super().__call__(*args, **kwargs)

    class Both(_Float, Watched):
        pass

    for cls, count in ((_Float, 0), (Both, 1)):
        q, x = _layer(cls)
        r = torch.ones(4, 16)
        assert torch.equal(q(x, residual=r), _float_forward(q, x, r)) and len(seen) == count
        with monkeypatch.context() as m:
            calls, real = [], torch.nn.Module.__call__
            m.setattr(torch.nn.Module, "__call__", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
            assert torch.equal(q(x, r), _float_forward(q, x, r)) and len(calls) == 1
        with pytest.raises(TypeError):
            q()
        seen.clear()
    with pytest.raises((TypeError, AttributeError)):
        QuantLinear.__call__(3)
    with pytest.raises(TypeError):
        QuantLinear.__call__()
