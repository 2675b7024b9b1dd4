"""CPU-only checks of the layer wrapper: constructor rules, parameter names and shapes
(state_dict compatibility with the reference), the initialisation recipe, error behaviour."""
import math
import os

import numpy as np
import pytest
import torch

from sru_amd.modules import SRU, SRUCell

HERE = os.path.dirname(os.path.abspath(__file__))


def test_loads_the_reference_state_dict_of_the_regression_artifact():
    z = np.load(os.path.join(HERE, "golden", "regression_2.3.5.npz"))
    kwargs = {k.split("/", 1)[1]: z[k].item() for k in z.files if k.startswith("kwargs/")}
    model = SRU(**kwargs)
    state = {k.split("/", 1)[1]: torch.tensor(z[k]) for k in z.files if k.startswith("state/")}
    assert set(model.state_dict()) == set(state)
    model.load_state_dict(state, strict=True)
    assert model.rnn_lst[0].num_matrices == 4 and model.rnn_lst[1].num_matrices == 3
    assert model.rnn_lst[0].dropout == pytest.approx(0.1) and model.rnn_lst[1].dropout == 0


@pytest.mark.parametrize("kw,keys", [
    (dict(input_size=8, hidden_size=8), {"weight", "weight_c", "bias", "scale_x"}),
    (dict(input_size=16, hidden_size=8, n_proj=4),
     {"weight", "weight_proj", "weight_c", "bias", "scale_x"}),
    (dict(input_size=8, hidden_size=8, layer_norm=True),
     {"weight", "weight_c", "bias", "scale_x", "layer_norm.weight", "layer_norm.bias"}),
])
def test_cell_parameter_names(kw, keys):
    assert set(SRUCell(**kw).state_dict()) == keys


def test_shape_rules():
    # k = 4 only when there is a skip term that cannot be the input itself (sru/modules.py:131-133)
    assert SRUCell(8, 8).num_matrices == 3
    assert SRUCell(8, 4, bidirectional=True).num_matrices == 3
    assert SRUCell(8, 8, bidirectional=True).num_matrices == 4
    assert SRUCell(6, 8, has_skip_term=False).num_matrices == 3
    # projection only when it is a bottleneck (sru/modules.py:126-128)
    assert SRUCell(16, 8, n_proj=8).projection_size == 0
    assert SRUCell(16, 8, n_proj=4).weight.shape == (4, 32)   # 16 != 8: four streams
    assert SRUCell(16, 8, n_proj=4).weight_proj.shape == (16, 4)
    cell = SRUCell(6, 5, bidirectional=True)
    assert cell.weight.shape == (6, 40) and cell.weight_c.shape == (20,) and cell.bias.shape == (20,)
    stack = SRU(6, 5, num_layers=3, bidirectional=True, dropout=0.2, proj_input_to_hidden_first=True)
    assert stack.input_to_hidden.weight.shape == (10, 6)
    assert [c.input_size for c in stack.rnn_lst] == [10, 10, 10]
    assert [c.dropout for c in stack.rnn_lst] == [0.2, 0.2, 0.0]
    # defaults differ between the two classes (sru/modules.py:41 vs :444)
    assert SRUCell(4, 4).rescale is True and SRU(4, 4).rnn_lst[0].rescale is False


def test_initialisation_recipe():
    torch.manual_seed(0)
    d = 256
    cell = SRUCell(d, d, highway_bias=-2.0, rescale=True)
    w = cell.weight.detach().view(d, 1, d, 3)
    assert abs(float(w[..., 0].var()) * d - 1.0) < 0.05          # Var = 1/d
    assert abs(float(w[..., 1].var()) * d - 0.5) < 0.03          # gate columns * sqrt(0.5)
    assert abs(float(w[..., 2].var()) * d - 0.5) < 0.03
    assert abs(float(cell.weight_c.var()) - 0.5) < 0.08          # Var = 1 then * 0.5
    assert torch.all(cell.bias[:d] == 0) and torch.all(cell.bias[d:] == -2.0)
    assert float(cell.scale_x) == pytest.approx(math.sqrt(1 + 2 * math.exp(-2.0)))
    assert float(SRUCell(d, d, rescale=False).scale_x) == 1.0
    # k = 4 with rescale: the fourth stream carries the scale (sru/modules.py:208-210)
    c4 = SRUCell(d, 2 * d, highway_bias=0.0, rescale=True)
    w4 = c4.weight.detach().view(d, 1, 2 * d, 4)
    assert abs(float(w4[..., 3].var()) * d - 3.0) < 0.15
    # layer norm shrinks the weights, dropout rescales the candidate stream
    cl = SRUCell(d, d, layer_norm=True, dropout=0.5)
    wl = cl.weight.detach().view(d, 1, d, 3)
    assert abs(float(wl[..., 0].var()) * d - 0.01 * 0.5) < 0.001
    v1 = SRUCell(d, d, v1=True)
    assert torch.all(v1.weight_c == 0) and not v1.weight_c.requires_grad
    assert float(SRUCell(d, d, weight_c_init=0.01).weight_c.abs().max()) <= 0.01


def test_error_behaviour():
    cell, stack = SRUCell(4, 4), SRU(4, 4)
    with pytest.raises(ValueError):
        cell(torch.zeros(2, 2, 2, 4))
    with pytest.raises(ValueError):
        stack(torch.zeros(3, 4))
    with pytest.raises(ValueError):
        stack(torch.zeros(3, 2, 4), c0=torch.zeros(2, 4))
    with pytest.raises(RuntimeError):          # no CPU path for the recurrence
        stack(torch.zeros(3, 2, 4))

    class Bad(torch.nn.Module):
        def forward(self, x):
            return x
    with pytest.raises(ValueError):
        SRUCell(4, 4, custom_m=Bad()).compute_UV(torch.zeros(3, 2, 4), None, None)


def test_repr_follows_the_reference_format():
    # sru/modules.py:384-419
    assert repr(SRUCell(8, 8)) == "SRUCell(8, 8, rescale=True)"
    cell = SRUCell(16, 8, dropout=0.1, rnn_dropout=0.2, bidirectional=True, n_proj=4, use_tanh=True,
                   highway_bias=-1.0, has_skip_term=False, layer_norm=True, rescale=False, v1=True)
    assert repr(cell) == ("SRUCell(16, 8, projection_size=4, dropout=0.1, rnn_dropout=0.2, bidirectional=True, "
                          "highway_bias=-1.0, activation=tanh, v1=True, rescale=False, has_skip_term=False, "
                          "layer_norm=True)")
    with_m = SRUCell(4, 4, custom_m=torch.nn.Linear(4, 12, bias=False))
    assert repr(with_m) == ("SRUCell(4, 4, rescale=True,\n  custom_m=Linear(in_features=4, out_features=12, "
                            "bias=False)\n)")
    assert "SRUCell(4, 4, rescale=False)" in repr(SRU(4, 4))


def _drop(module, name):
    """Removes an attribute wherever nn.Module keeps it (plain attribute or sub-module slot)."""
    if name in module._modules:
        del module._modules[name]
    else:
        module.__dict__.pop(name, None)


def test_make_backward_compatible():
    # sru/modules.py:660-689: attribute names of releases <= 2.1.7 and <= 2.1.9
    model = SRU(6, 5, num_layers=2, bidirectional=True, projection_size=2)
    # an object as release 2.1.7 pickled it: old names only
    old = SRU(6, 5, num_layers=2, bidirectional=True, projection_size=2)
    old.n_in, old.n_out, old.out_size, old.depth, old.n_proj = 6, 5, 10, 2, 2
    old.ln_lst, old.use_weight_norm = [], False
    for name in ("input_size", "hidden_size", "output_size", "num_layers", "projection_size", "use_layer_norm",
                 "nn_rnn_compatible_return"):
        delattr(old, name)
    _drop(old, "input_to_hidden")
    for cell in old.rnn_lst:
        cell.n_in, cell.n_out, cell.k, cell.n_proj = cell.input_size, cell.hidden_size, cell.num_matrices, 2
        for name in ("input_size", "hidden_size", "output_size", "num_matrices", "projection_size", "custom_m",
                     "layer_norm"):
            _drop(cell, name)
    old.make_backward_compatible()
    for name in ("input_size", "hidden_size", "output_size", "num_layers", "projection_size"):
        assert getattr(old, name) == getattr(model, name), name
    assert old.use_layer_norm is False and old.nn_rnn_compatible_return is False
    assert old.input_to_hidden is None
    for cell, new in zip(old.rnn_lst, model.rnn_lst):
        for name in ("input_size", "hidden_size", "output_size", "num_matrices", "projection_size"):
            assert getattr(cell, name) == getattr(new, name), name
        assert cell.layer_norm is None and cell.custom_m is None
    # what cannot be carried over is refused
    old.use_weight_norm = True
    with pytest.raises(Exception, match="Weight norm"):
        old.make_backward_compatible()
    old.use_weight_norm, old.ln_lst = False, [1]
    with pytest.raises(Exception, match="Layer norm"):
        old.make_backward_compatible()
    old.ln_lst = []
    old.rnn_lst[0].activation_type = 2
    with pytest.raises(Exception, match="ReLU or SeLU"):
        old.make_backward_compatible()
    # a current object passes through unchanged
    before = dict(model.__dict__)
    model.make_backward_compatible()
    assert {k: v for k, v in model.__dict__.items() if k != "_modules"} == \
        {k: v for k, v in before.items() if k != "_modules"}


def test_large_stack_restatement_equals_the_python_loop_restatement():
    # tests/stack_ref.py: the float64 stack built on the C oracle (used at sizes where the Python
    # loop is too slow) must agree with the one built on the differentiable torch loop
    from tests.stack_ref import stack_forward, stack_forward_large
    torch.manual_seed(4)
    model = SRU(6, 8, num_layers=3, bidirectional=True, layer_norm=True, rescale=True, projection_size=3,
                dropout=0.2)
    x = torch.randn(9, 4, 6)
    pad = torch.arange(9)[:, None] >= torch.tensor([9, 4, 7, 1])[None, :]
    h1, c1, p1 = stack_forward(model, x, mask_pad=pad)
    h2, c2, p2 = stack_forward_large(model, x, mask_pad=pad, device="cpu")
    probe = torch.randn(h1.shape, dtype=torch.float64)
    (h1 * probe).sum().backward()
    (h2 * probe).sum().backward()
    assert float((h1 - h2).abs().max()) <= 1e-12 and float((c1 - c2).abs().max()) <= 1e-12
    for n in p1:
        assert float((p1[n].grad - p2[n].grad).abs().max()) <= 1e-10 * max(1.0, float(p1[n].grad.abs().max())), n


class _Own(Exception):
    pass


def _own_step(*args):
    raise _Own


@pytest.mark.parametrize("step", ["compute_U", "compute_UV", "apply_recurrence"])
@pytest.mark.parametrize("where", ["instance", "class", "subclass"])
def test_a_step_put_in_place_of_the_layers_own_is_called(where, step, monkeypatch):
    """The one-kernel route of 16-bit layers stands for the layer's own steps only."""
    from sru_amd import modules
    cls = type("Derived", (SRUCell,), {step: _own_step}) if where == "subclass" else SRUCell
    cell = cls(64, 64).half()
    x = torch.zeros(1, 2, 64).half()
    route = (torch.ones(1, 2, 64), torch.ones(2, 64))
    monkeypatch.setattr(modules, "layer_forward", lambda *a: route)
    if where != "subclass":
        with torch.no_grad():
            assert cell(x) == route
        monkeypatch.setattr(cell if where == "instance" else SRUCell, step, _own_step, raising=True)
    with torch.no_grad(), pytest.raises(_Own):
        cell(x)


@pytest.mark.parametrize("step", ["forward", "backward", "apply"])
def test_a_step_put_in_place_of_the_recurrences_own_is_called(step, monkeypatch):
    """A layer's node of native code stands for the Function as this package defines it."""
    from sru_amd import ElementwiseRecurrence, _lib
    cell, x = SRUCell(8, 8), torch.zeros(2, 2, 8)
    node = (torch.ones(2, 2, 8), torch.ones(2, 8))
    monkeypatch.setattr(_lib, "host", lambda: type("Host", (), {"layer": staticmethod(lambda *a: node)}))
    assert cell._native_layer(x, x, None, cell.scale_x, None, None) is node
    monkeypatch.setattr(ElementwiseRecurrence, step, staticmethod(_own_step))
    assert cell._native_layer(x, x, None, cell.scale_x, None, None) is None


@pytest.mark.parametrize("name", ["__call__", "_call_impl", "forward", "compute_U", "apply_recurrence"])
def test_a_stack_in_one_call_stands_for_cells_as_torch_calls_them(name, monkeypatch):
    from sru_amd import _lib
    model, x = SRU(8, 8).bfloat16(), torch.zeros(2, 2, 8).bfloat16()
    monkeypatch.setattr(_lib, "host", lambda: type("Host", (), {"stack_forward": staticmethod(lambda *a: "whole")}))
    with torch.no_grad():
        assert model._whole_stack(x, None, None) == "whole"
        own = getattr(SRUCell, name)
        monkeypatch.setattr(torch.nn.Module if name.startswith("_") else SRUCell, name, lambda self, *a, **kw: own(self, *a, **kw))
        assert model._whole_stack(x, None, None) is None


@pytest.mark.parametrize("kind,asked", [("plain", True), ("16-bit", False), ("frozen", False), ("frozen, the input's gradient", True), ("frozen, the state's gradient", True),
                                        ("a replica's", True)])
def test_a_layers_node_is_asked_for_where_it_can_be(kind, asked, monkeypatch):
    from sru_amd import _lib
    cell, x, c0, calls = SRUCell(8, 8), torch.zeros(2, 2, 8), torch.zeros(2, 8), []
    if kind == "16-bit":
        cell, x = cell.bfloat16(), x.bfloat16()
    cell.requires_grad_("frozen" not in kind)
    x.requires_grad_("input" in kind)
    c0.requires_grad_("state" in kind)
    if "replica" in kind:        # (torch.nn.DataParallel gives it its parameters as attributes)
        for name, p in list(cell._parameters.items()):
            del cell._parameters[name]
            cell.__dict__[name] = p
    monkeypatch.setattr(_lib, "host", lambda: type("Host", (), {"layer": staticmethod(lambda *a: calls.append(1))}))
    assert cell._native_layer(x, x, c0, cell.scale_x, None, None) is None
    assert bool(calls) == asked


def test_what_is_never_a_stack_is_not_looked_at():
    """A layer by itself, float weights and calls with gradients: asking costs a fifth of a single layer's step."""
    looked = []

    class Watched(SRU):
        def __getattr__(self, name):
            looked.append(name)
            return super().__getattr__(name)

    for layers, dtype, grad in ((1, torch.bfloat16, False), (2, torch.float32, False), (2, torch.bfloat16, True), (2, torch.bfloat16, False)):
        model, x = Watched(8, 8, num_layers=layers).to(dtype), torch.zeros(1, 2, 8, dtype=dtype)
        looked.clear()
        with torch.set_grad_enabled(grad):
            assert model._whole_stack(x, None, None) is None    # (host tensors)
        assert looked == []


@pytest.mark.parametrize("change", [None, lambda m: setattr(m, "num_layers", 2), lambda m: m.rnn_lst.append(SRUCell(8, 8))])
def test_a_stack_in_one_call_has_as_many_layers_as_run_one_by_one(change, monkeypatch):
    from sru_amd import _lib
    model = SRU(8, 8, num_layers=3).bfloat16()
    if change is not None:
        change(model)
    x = torch.zeros(2, 2, 8).bfloat16()
    called = []
    monkeypatch.setattr(_lib, "host", lambda: type("Host", (), {"stack_forward": staticmethod(lambda cells, *a: ("h", len(cells)))}))
    for cell in model.rnn_lst:
        monkeypatch.setattr(cell, "forward", lambda x, state, mask_pad=None: (called.append(1) or x, x[0]))
    with torch.no_grad():
        assert model._whole_stack(x, None, None) == (("h", 3) if change is None else None)
        model(x)
    assert len(called) == {None: 0}.get(change, model.num_layers)


def test_native_calls_stand_aside_under_modes():
    """Under a mode that sees every call the native host code leaves the call to Python."""
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    from sru_amd import _lib
    x, w, wc = torch.zeros(1, 2, 64).half(), torch.zeros(64, 192).half(), torch.zeros(128).half()
    call = lambda: _lib.host().layer_forward(x, x, None, w, wc, wc, None, 0, 64, False, True, None, None)
    assert call() is None                  # (host tensors: for the general way to look at)
    with FlopCounterMode(display=False):
        assert call() is False
    with TorchFunctionMode():
        assert call() is False
    # (a default device is a mode, too, but watches nothing)
    with torch.device("cpu"):
        assert call() is None
        with TorchFunctionMode():
            assert call() is False
    assert call() is None


class _Scaled(torch.Tensor):
    """Eight-bit values and a scale that show themselves as a 16-bit tensor without memory."""
    @staticmethod
    def __new__(cls, values, scale):
        out = torch.Tensor._make_wrapper_subclass(cls, values.shape, dtype=torch.bfloat16)
        out.values, out.scale = values, scale
        return out

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        return func(*[(a.values * a.scale).bfloat16() if isinstance(a, cls) else a for a in args], **(kwargs or {}))


def test_small_tensors_of_other_types_are_converted():
    """What a 16-bit small tensor of a subclass holds comes from its own conversion, never from its memory."""
    from sru_amd import functional
    L, B, d = 3, 2, 4
    pb = functional._problem_cached(torch.bfloat16, 3, L, B, L * B * d * 3, d * 3, 0, d, False, True, 0, False, False, False)
    u, x, wc = torch.zeros(L, B, 3 * d).bfloat16(), torch.zeros(L, B, d).bfloat16(), torch.ones(2 * d).bfloat16()
    bias = _Scaled(torch.arange(2 * d, dtype=torch.int8), 0.5)
    (_, _, wc_, bias_, *_), small16 = functional._prepare_inputs(pb, u, x, wc, bias, None, None, None, None, narrow_small=True)
    assert small16 == functional._lib.SMALL_WEIGHT_C and wc_.dtype == torch.bfloat16
    assert type(bias_) is torch.Tensor and bias_.dtype == torch.float32
    assert torch.equal(bias_, 0.5 * torch.arange(2 * d))


@pytest.mark.parametrize("which", [7, 8])
def test_flags_without_a_truth_value_are_refused_by_the_general_way(which):
    from sru_amd import elementwise_recurrence_forward
    args = [torch.zeros(2, 2, 12), torch.zeros(2, 2, 4), torch.zeros(8), torch.zeros(8), None, 0, 4, False, True]
    args[which] = torch.zeros(2)
    with pytest.raises(RuntimeError):      # (host tensors here; with device tensors the flag itself)
        elementwise_recurrence_forward(*args, keep_c=False)


def test_a_layers_product_can_be_traced():
    """With the tracer's own check, which repeats the call without gradients and compares line by line."""
    from sru_amd.functional import dense
    x, w = torch.randn(5000, 64), torch.randn(64, 192, requires_grad=True)
    traced = torch.jit.trace(dense, (x, w))
    assert torch.equal(traced(x[:7], w), x[:7] @ w)
