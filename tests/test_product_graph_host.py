"""The layer product's place in torch's graphs (functional.dense, functional._Product), on the CPU: which gradients a
backward pass makes."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from sru_amd import functional


class CountProducts(TorchDispatchMode):
    """Counts matrix products; as a mode that watches, it has the weight's gradient made by torch."""

    def __init__(self):
        super().__init__()
        self.count = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.count += func is torch.ops.aten.mm.default
        return func(*args, **(kwargs or {}))


REQUESTS = {
    "backward": (lambda y, x, w: y.backward(), 2),
    "input": (lambda y, x, w: torch.autograd.grad(y, x), 1),
    "weight": (lambda y, x, w: torch.autograd.grad(y, w), 1),
    "both": (lambda y, x, w: torch.autograd.grad(y, (x, w)), 2),
    "inputs=input": (lambda y, x, w: y.backward(inputs=[x]), 1),
    "inputs=weight": (lambda y, x, w: y.backward(inputs=[w]), 1),
    "input, to differentiate again": (lambda y, x, w: torch.autograd.grad(y, x, create_graph=True), 1),
}


@pytest.mark.parametrize("request_name", list(REQUESTS))
@pytest.mark.parametrize("leaf", [True, False])
@pytest.mark.parametrize("converted", [True, False])
def test_gradients_that_nobody_asked_for_are_not_made(request_name, leaf, converted):
    request, products = REQUESTS[request_name]
    gen = torch.Generator().manual_seed(1)
    w = torch.randn(6, 9, generator=gen).requires_grad_()
    got = []
    for own in (True, False):
        x = torch.randn(5, 6, generator=gen.manual_seed(2)).requires_grad_()
        y = x if leaf else 2 * x
        narrow = w.bfloat16() if converted else w
        out = (functional._Product.apply(y.to(narrow.dtype), narrow, w if converted else None) if own
               else y.to(narrow.dtype).mm(narrow)).float().sum()
        w.grad = None
        with CountProducts() as products_of_pass:
            grads = request(out, x if leaf or "inputs=" in request_name else y, w)
        got.append([t for t in (grads or (x.grad, w.grad))])
        assert products_of_pass.count == products
    for a, b in zip(*got):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("rows", [100, 5000])
def test_a_product_is_compiled_whole(rows, grad):
    torch._dynamo.reset()
    x, w = torch.randn(rows, 64), torch.randn(64, 192, requires_grad=True)
    with torch.set_grad_enabled(grad):
        assert torch.equal(torch.compile(functional.dense, backend="eager", fullgraph=True)(x, w), x @ w)


def test_a_default_device_watches_nothing():
    from torch.overrides import TorchFunctionMode
    assert not functional._observed()
    with torch.device("cpu"):
        assert not functional._observed()
        with CountProducts():
            assert functional._observed()
        with TorchFunctionMode():
            assert functional._observed()
    with torch.autograd.forward_ad.dual_level():
        assert functional._observed()
    seen = []
    torch.func.vmap(lambda t: seen.append(functional._observed()) or t)(torch.zeros(2))
    torch.jit.trace(lambda t: seen.append(functional._observed()) or t + 1, torch.zeros(2), check_trace=False)
    assert seen == [True, True] and not functional._observed()
