"""The weight gradient of a layer's dense product over many rows (csrc/product_grad.hip): by itself against float64, and
through the layer against torch's own product."""
import ctypes

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from sru_amd import SRUCell, _lib, functional

pytestmark = pytest.mark.gpu

CODE = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}
HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
# (rows, inner, cols): both tiles, whole and cut off at either edge, rows with a remainder of one piece and of none, walks
# of uneven parts down to four tiles of rows
SIZES = [(4096, 512, 1536), (8193, 128, 2048), (8255, 136, 2056), (8256, 520, 1000), (8200, 264, 1032), (5000, 1024, 2880), (8196, 2048, 128),
         (3000, 512, 3072), (8192, 128, 384), (6000, 1000, 3000), (8196, 456, 6008)]
WIDE = [(5000, 1024, 2880), (6000, 1000, 3000), (8196, 456, 6008)]    # in tiles of 192 columns


@pytest.mark.parametrize("out", [torch.float32, "narrow"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,inner,cols", SIZES)
def test_gradient(rows, inner, cols, dtype, out):
    out = dtype if out == "narrow" else out
    gen = torch.Generator().manual_seed(rows + cols)
    x, g = torch.randn(rows, inner, generator=gen).to(dtype), torch.randn(rows, cols, generator=gen).to(dtype)
    xd, gd = x.cuda(), g.cuda()
    lib, p = _lib.load(), lambda t: ctypes.c_void_p(t.data_ptr())
    nbytes = lib.sru_amd_product_grad_workspace_bytes(CODE[dtype], rows, inner, cols)
    assert nbytes > 0 and nbytes % (4 * inner * cols) == 0
    work = torch.full((nbytes // 4 + 64,), float("nan"), device="cuda")
    got = torch.full((inner + 1, cols), float("nan"), device="cuda", dtype=out)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        rc = lib.sru_amd_product_grad(CODE[dtype], rows, inner, cols, p(xd), p(gd), CODE[out], p(got), p(work), ctypes.c_size_t(nbytes),
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
    assert rc == 0
    kernels = [e.name for e in seen.events() if "product_grad<" in e.name]
    assert len(kernels) == 1 and ("_bits, 3>" in kernels[0]) == ((rows, inner, cols) in WIDE)
    assert torch.isnan(got[inner]).all() and torch.isnan(work[nbytes // 4:]).all()
    want = x.double().t() @ g.double()
    # float sums of `rows` terms whose rounding errors are independent (ten deviations), then the result's rounding
    spread = (x.double().square().t() @ g.double().square()).sqrt()
    bound = 10 * rows ** 0.5 * 2.0 ** -24 * spread + HALF_ULP[out] * want.abs()
    assert ((got[:inner].cpu().double() - want).abs() <= bound).all()


def layer_gradients(cell, x, probe, autocast, **kw):
    cell.zero_grad(set_to_none=True)
    x = x.detach().requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        h, _ = cell(x)
    h.backward(probe.to(h.dtype), **kw)
    return {"x": x.grad, **{n: p.grad for n, p in cell.named_parameters()}}


@pytest.mark.parametrize("autocast,inp,d,kw", [(True, 512, 512, {}), (True, 1024, 1024, dict(n_proj=512)), (False, 512, 512, {}),
                                              (True, 520, 512, {}), (True, 512, 512, dict(layer_norm=True))])
def test_layer(autocast, inp, d, kw, monkeypatch):
    torch.manual_seed(1)
    cell = SRUCell(inp, d, **kw).cuda()
    if not autocast:
        cell = cell.bfloat16()
    x = torch.randn(260, 33, inp, device="cuda").to(cell.weight.dtype)
    probe = torch.randn(260, 33, d, device="cuda")
    calls, original = [], functional._weight_gradient
    monkeypatch.setattr(functional, "_weight_gradient", lambda *a: calls.append(1) or original(*a))
    got = layer_gradients(cell, x, probe, autocast)
    assert len(calls) == (2 if "n_proj" in kw else 1)
    monkeypatch.setattr(functional, "_grad_workspace", lambda *a: 0)
    want = layer_gradients(cell, x, probe, autocast)
    assert len(calls) == (2 if "n_proj" in kw else 1)
    for name in want:
        assert got[name].dtype == want[name].dtype
        if name in ("weight", "weight_proj"):
            # torch's is rounded to 16 bits on its way: half a unit in the last place, 2^-8 of a value at the most;
            # where ours is rounded as well the two may be a whole unit apart
            err = (got[name].double() - want[name].double()).abs()
            assert (err <= (2.0 ** -8 if autocast else 2.0 ** -7) * want[name].abs().double() + 1e-4 * want[name].abs().max().double()).all(), name
        else:
            assert torch.equal(got[name], want[name]), name


def test_forms_that_keep_torchs_product():
    from torch.utils.flop_counter import FlopCounterMode
    cell = SRUCell(512, 512).cuda().bfloat16()
    x = torch.randn(4096, 512, device="cuda").bfloat16().requires_grad_()
    name = lambda t: type(t.grad_fn).__name__
    assert name(functional.dense(x, cell.weight)) == "_ProductBackward"
    assert name(functional.dense(x[:3800], cell.weight)) == "MmBackward0"
    assert name(functional.dense(x, cell.weight.detach())) == "MmBackward0"
    with FlopCounterMode(display=False) as flops:
        functional.dense(x, cell.weight).sum().backward()
    assert flops.get_total_flops() == 3 * 2 * 4096 * cell.weight.numel()
    with torch.autograd.forward_ad.dual_level():
        out = functional.dense(torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x)), cell.weight)
        assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None
    assert torch.func.vmap(lambda t: functional.dense(t, cell.weight))(torch.stack([x.detach()] * 2)).shape == (2, 4096, 1536)
    with pytest.raises(RuntimeError):
        functional.dense(x[:, :504], cell.weight)


def test_twice_differentiable():
    x = torch.randn(8192, 512, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(512, 512, device="cuda").requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = functional.dense(x, w)
        plain = x.mm(w)
    v = torch.randn_like(out).requires_grad_()
    for a, b in zip(*(torch.autograd.grad(torch.autograd.grad(o, (x, w), v, create_graph=True), (v, w, x), [torch.ones_like(x), torch.ones_like(w)])
                      for o in (out, plain))):
        assert torch.equal(a, b)


def test_strided_gradient_saved_tensor_hooks_and_a_stepped_weight():
    x = torch.randn(8192, 512, device="cuda").bfloat16()
    w = torch.randn(512, 512, device="cuda").requires_grad_()
    v = torch.randn(512, 8192, device="cuda").bfloat16().t()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
            out = functional.dense(x, w)
    want = (x.double().t() @ v.double()).float()
    with torch.no_grad():
        w.add_(1.0)                 # (the products keep their own 16-bit weight)
    out.backward(v)
    assert ((w.grad - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max()).all()


def test_in_a_graph():
    x, g = torch.randn(4096, 512, device="cuda").bfloat16(), torch.randn(4096, 1536, device="cuda").bfloat16()
    functional._weight_gradient(x, g, torch.float32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = functional._weight_gradient(x, g, torch.float32)
    for _ in range(4):
        x.copy_(torch.randn_like(x))
        graph.replay()
        replayed = out.clone()
        assert torch.equal(replayed, functional._weight_gradient(x, g, torch.float32))


def test_the_inputs_gradient_alone(monkeypatch):
    cell = SRUCell(512, 512).cuda().bfloat16()
    x = torch.randn(260, 32, 512, device="cuda").bfloat16().requires_grad_()
    calls, original = [], functional._weight_gradient
    monkeypatch.setattr(functional, "_weight_gradient", lambda *a: calls.append(1) or original(*a))
    h, _ = cell(x)
    only, = torch.autograd.grad(h, x, torch.ones_like(h), retain_graph=True)
    assert not calls
    both = torch.autograd.grad(h, (x, cell.weight), torch.ones_like(h))
    assert len(calls) == 1 and torch.equal(only, both[0])


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("rows", [640, 8192])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_compiled_whole(dtype, rows, grad):
    torch._dynamo.reset()
    x, w = torch.randn(rows, 128, device="cuda").to(dtype), torch.randn(128, 384, device="cuda").to(dtype).requires_grad_()
    with torch.set_grad_enabled(grad):
        assert torch.equal(torch.compile(functional.dense, backend="eager", fullgraph=True)(x, w), x @ w)


def test_a_weight_is_converted_once_in_an_autocast_region():
    x, w = torch.randn(8192, 512, device="cuda"), torch.randn(512, 512, device="cuda").requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        outs = [functional.dense(x, w) for _ in range(2)]
        kept = [o.grad_fn.saved_tensors[1].data_ptr() for o in outs]
        assert kept[0] == kept[1]
        with torch.autocast("cuda", dtype=torch.bfloat16, cache_enabled=False):
            other = functional.dense(x, w)
            assert other.grad_fn.saved_tensors[1].data_ptr() != kept[0]
    torch.autograd.backward(outs, [torch.ones_like(o) for o in outs])
    twice, w.grad = w.grad, None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        functional.dense(x, w).backward(torch.ones_like(outs[0]))
    assert torch.equal(twice, 2 * w.grad)


@pytest.mark.parametrize("again", [False, True])
def test_a_weight_converted_without_gradients_earlier_in_the_region(again):
    x, w = torch.randn(8192, 512, device="cuda"), torch.randn(512, 512, device="cuda").requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        with torch.no_grad():
            functional.dense(x, w)
        out = functional.dense(x, w)
    got, = torch.autograd.grad(out, w, torch.ones_like(out), create_graph=again)
    want = x.bfloat16().double().t() @ torch.ones_like(out).double()
    # a sum of 8192 rounded once to 16 bits, or none but its own float sums
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max()).all()


def test_a_default_device_changes_nothing():
    x, w = torch.randn(8192, 512, device="cuda").bfloat16(), torch.randn(512, 512, device="cuda").bfloat16().requires_grad_()
    floats = torch.randn(640, 128, device="cuda"), torch.randn(128, 384, device="cuda")
    with torch.device("cuda"):
        assert type(functional.dense(x, w).grad_fn).__name__ == "_ProductBackward"
        with torch.no_grad():
            assert functional._short_product(*floats) is not None


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,inner,cols", [(3001, 1416, 2984), (4096, 1032, 3648), (8225, 520, 9216)])
def test_rows_in_one_part(rows, inner, cols, out):
    """Tiles that fill the chip by themselves: an odd and an even number of tiles of rows, cut-off tiles at every edge; a
    float result is written by the product itself."""
    gen = torch.Generator().manual_seed(rows)
    x, g = (torch.randn(rows, n, generator=gen).bfloat16().cuda() for n in (inner, cols))
    assert functional._grad_workspace(x.dtype, rows, inner, cols) == 4 * inner * cols
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        got = functional._weight_gradient(x, g, out)
        torch.cuda.synchronize()
    assert any("product_grad<" in e.name for e in seen.events())
    assert any("add_slices<" in e.name for e in seen.events()) == (out != torch.float32)
    want, spread = x.double().t() @ g.double(), (x.double().square().t() @ g.double().square()).sqrt()
    # (as above: independent rounding errors of `rows` float sums, then the result's rounding)
    assert ((got.double() - want).abs() <= 10 * rows ** 0.5 * 2.0 ** -24 * spread + HALF_ULP[out] * want.abs()).all()
