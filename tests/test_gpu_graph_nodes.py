"""A layer with gradients as one node of the native host code against the same layer through torch's products and the
recurrence's own Function."""
import threading

import pytest
import torch

from sru_amd import SRU, ElementwiseRecurrence, SRUCell, functional

pytestmark = pytest.mark.gpu

# input, hidden, constructor arguments, autocast, parameter and input types
FORMS = [(64, 64, {}, False, torch.float32), (48, 64, {}, False, torch.float32), (128, 64, dict(bidirectional=True, n_proj=32), False, torch.float32),
         (64, 64, dict(use_tanh=True, dropout=0.3), False, torch.float32), (64, 64, dict(has_skip_term=False), False, torch.float32),
         (65, 65, dict(rescale=False), False, torch.float32), (64, 64, dict(layer_norm=True), False, torch.float32),
         (64, 64, {}, True, torch.float32), (64, 64, {}, True, torch.bfloat16), (96, 64, dict(n_proj=32), True, torch.bfloat16),
         (128, 64, dict(bidirectional=True, n_proj=32), True, torch.bfloat16), (64, 64, dict(layer_norm=True), True, torch.bfloat16),
         (512, 512, dict(n_proj=128), True, torch.bfloat16), (64, 64, {}, False, torch.bfloat16)]


def one_pass(cell, x, c0, pad, probe, probe_c, autocast, seed=7):
    leaves = [x.detach().requires_grad_(), c0.detach().requires_grad_()]
    cell.zero_grad()
    torch.manual_seed(seed)      # (of the dropout mask)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        h, c = cell(leaves[0], leaves[1], mask_pad=pad)
    name = h.grad_fn.name()
    torch.autograd.backward([h, c], [probe.to(h.dtype), probe_c.to(c.dtype)])
    return name, {"h": h.detach(), "c": c.detach(), "x": leaves[0].grad, "c0": leaves[1].grad, **{n: p.grad.clone() for n, p in cell.named_parameters()}}


@pytest.mark.parametrize("inp,d,kw,autocast,x_dtype", FORMS)
@pytest.mark.parametrize("rows", [(7, 3), (130, 32)])
def test_gradients(rows, inp, d, kw, autocast, x_dtype, monkeypatch):
    torch.manual_seed(inp)
    L, B = rows
    cell = SRUCell(inp, d, **kw).cuda()
    plain = autocast or x_dtype == torch.float32      # (small tensors in 16 bits go the general way)
    if not plain:
        cell = cell.to(x_dtype)
    x = torch.randn(L, B, inp, device="cuda").to(x_dtype)
    c0 = torch.randn(B, cell.output_size, device="cuda")
    pad = torch.rand(L, B, device="cuda") < 0.2
    probe, probe_c = torch.randn(L, B, cell.output_size, device="cuda"), torch.randn(B, cell.output_size, device="cuda")
    name, got = one_pass(cell, x, c0, pad, probe, probe_c, autocast)
    assert (name == "SRULayerBackward") == plain
    monkeypatch.setattr(functional, "replaced", lambda: True)
    name, want = one_pass(cell, x, c0, pad, probe, probe_c, autocast)
    assert name == "ElementwiseRecurrenceBackward"
    # Float: other orders of summation, 2^-23 of a sum's largest terms times the square root of their number, carried on through the
    # walk. 16 bits: the skip term's and the product's gradient are rounded once instead of twice, a weight's not on its
    # way to float, and a product of another kernel may round U to its neighbour: units of 2^-8 of the largest values around.
    unit = 2.0 ** -7 if autocast else 2e-5
    for n in want:
        assert got[n].dtype == want[n].dtype and got[n].shape == want[n].shape
        error = (got[n].double() - want[n].double()).abs().max() / want[n].double().abs().max().clamp(min=1e-6)
        assert float(error) <= unit, (n, float(error))


def test_graph_properties():
    cell = SRUCell(64, 64, n_proj=32).cuda()
    x = torch.randn(9, 4, 64, device="cuda").requires_grad_()
    h, c = cell(x)
    probe = torch.randn_like(h)
    full = torch.autograd.grad(h, (x, cell.weight, cell.weight_proj, cell.weight_c), probe, retain_graph=True)
    for i, leaf in enumerate((x, cell.weight, cell.weight_proj, cell.weight_c)):      # one at a time, and again
        assert torch.equal(torch.autograd.grad(h, leaf, probe, retain_graph=True)[0], full[i])
    assert torch.autograd.grad(c.sum(), x, retain_graph=True)[0].shape == x.shape     # the last state alone
    assert torch.equal(torch.autograd.grad(h, x, probe.transpose(0, 1).contiguous().transpose(0, 1))[0], full[0])   # a strided gradient
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(h, x, probe)
    h, _ = cell(x)
    kept = cell.weight.detach().clone()
    with torch.no_grad():
        cell.weight.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(h, x, probe)
    with torch.no_grad():
        cell.weight.copy_(kept)
    with torch.autograd.graph.save_on_cpu():
        h, _ = cell(x)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(h, (x, cell.weight), probe), full))
    back = lambda v: v.transpose(0, -1).contiguous().transpose(0, -1) if v.dim() > 1 else v
    with torch.autograd.graph.saved_tensors_hooks(lambda v: v.clone(), back):         # other strides
        h, _ = cell(x)
    for a, b in zip(torch.autograd.grad(h, (x, cell.weight), probe), full):
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
    seen = []
    x.register_hook(seen.append)
    cell(x)[0].backward(probe)
    assert torch.equal(seen[0], x.grad) and float((seen[0] - full[0]).abs().max()) <= 1e-5 * float(full[0].abs().max())
    from torch.utils.checkpoint import checkpoint
    again = torch.autograd.grad(checkpoint(lambda t: cell(t)[0], x, use_reentrant=False), x, probe)[0]
    assert float((again - full[0]).abs().max()) <= 1e-5 * float(full[0].abs().max())


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("kw", [{}, dict(n_proj=128)])
def test_memory_of_a_backward_pass(kw, autocast, monkeypatch):
    """What the recurrence's part has read is free before the products' results are made, as where they are nodes of their own; with the graph kept
    it stays."""
    cell, x = SRUCell(1024, 1024, **kw).cuda(), torch.randn(64, 64, 1024, device="cuda").requires_grad_()
    with torch.no_grad():
        probe = torch.randn(64, 64, 1024, device="cuda").to(torch.bfloat16 if autocast else torch.float32)
    leaves = [x, *cell.parameters()]

    def peak(keep=False):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            h, _ = cell(x)
        torch.cuda.reset_peak_memory_stats()
        grads = torch.autograd.grad(h, leaves, probe, retain_graph=keep)
        most = torch.cuda.max_memory_allocated()
        if keep:
            assert all(torch.equal(a, b) for a, b in zip(grads, torch.autograd.grad(h, leaves, probe)))
        return most

    peak(), peak(True)
    node = peak()
    monkeypatch.setattr(functional, "replaced", lambda: True)
    peak()
    assert node <= peak() + (2 << 20)     # (allocations are rounded)


def test_a_backward_pass_that_a_mode_watches_shows_its_products():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Products(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen += func in (torch.ops.aten.mm.default, torch.ops.aten.addmm_.default)
            return func(*args, **(kwargs or {}))

    cell, x = SRUCell(512, 512, n_proj=128).cuda(), torch.randn(256, 32, 512, device="cuda").bfloat16().requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        h, _ = cell(x)
    assert h.grad_fn.name() == "SRULayerBackward" and functional._grad_workspace(torch.bfloat16, 8192, 512, 128) > 0
    probe, leaves = torch.randn_like(h), (x, cell.weight, cell.weight_proj)
    want = torch.autograd.grad(h, leaves, probe, retain_graph=True)
    with Products() as products:
        got = torch.autograd.grad(h, leaves, probe)
    assert products.seen == 4     # of two weights, of what was projected and of the input
    for a, b in zip(got, want):   # (a weight's is rounded to 16 bits on the way here)
        assert a.dtype == b.dtype and float((a.float() - b.float()).abs().max()) <= 2.0 ** -7 * float(b.float().abs().max())


@pytest.mark.parametrize("kw", [{}, dict(n_proj=32)])
def test_what_is_differentiable_twice_stays_so(kw, monkeypatch):
    """The dense products are, the recurrence's gradients are constants."""
    cell = SRUCell(64, 64, **kw).cuda()
    x = torch.randn(9, 4, 64, device="cuda").requires_grad_()
    probe, v = torch.randn(9, 4, 64, device="cuda"), torch.randn(9, 4, 64, device="cuda")

    def twice():
        leaves = list(cell.parameters())[:2 if kw else 1]
        first = torch.autograd.grad(cell(x)[0], [x] + leaves, probe, create_graph=True)
        total = (first[0] * v).sum() + sum((g * g.detach()).sum() for g in first[1:])
        return torch.autograd.grad(total, [x] + leaves, allow_unused=True)

    got = twice()
    monkeypatch.setattr(functional, "replaced", lambda: True)
    for a, b in zip(got, twice()):
        assert (a is None) == (b is None)
        assert a is None or float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


def test_threads():
    cell = SRUCell(64, 64).cuda()
    x = torch.randn(33, 8, 64, device="cuda")
    probe = torch.randn(33, 8, 64, device="cuda")
    want, results = torch.autograd.grad(cell(x)[0], cell.weight, probe)[0], []
    torch.cuda.synchronize()

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                results.append(torch.equal(torch.autograd.grad(cell(x)[0], cell.weight, probe)[0], want))

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 120 and all(results)


def test_compiled():
    torch._dynamo.reset()
    model = SRU(64, 64, num_layers=2, projection_size=16).cuda()
    x = torch.randn(20, 4, 64, device="cuda")
    run = lambda m: torch.autograd.grad(m(x)[0].sum(), list(model.parameters()))
    for a, b in zip(run(torch.compile(model, backend="eager")), run(model)):
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
    leaves = [torch.randn(10, 4, n, device="cuda").requires_grad_() for n in (192, 64)] + [torch.randn(128, device="cuda") for _ in range(2)]
    f = lambda u, s, w, b: ElementwiseRecurrence.apply(u, s, w, b, None, 0, 64, False, True, None, None, None)[0]
    assert torch.equal(torch.compile(f, backend="eager")(*leaves), f(*leaves))
