"""One time step of a whole stack in one launch (sru_amd_stack_forward) against the same layers called one by one, which
test_gpu_layer_forward.py holds against float64."""
import threading

import pytest
import torch

from sru_amd import SRU, modules

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def make(d, dtype, layers=3, **kw):
    torch.manual_seed(d + layers)
    model = SRU(d * (2 if kw.get("bidirectional") else 1), d, num_layers=layers, rescale=True, highway_bias=-0.5, **kw).cuda().to(dtype).eval()
    with torch.no_grad():
        for cell in model.rnn_lst:
            cell.bias += 0.3 * torch.randn_like(cell.bias)
    return model


def one_by_one(model, *args, **kw):
    original = modules.layer_forward
    modules.layer_forward = lambda *a: original(*a)
    try:
        return model(*args, **kw)
    finally:
        modules.layer_forward = original


def check(model, x, c0=None, pad=None):
    with torch.no_grad():
        assert model._whole_stack(x, c0, pad) is not None
        h, c = model(x, c0, mask_pad=pad)
        want_h, want_c = one_by_one(model, x, c0, mask_pad=pad)
    # the same sums in the same order, up to where the compiler contracts a product and a sum: a result may
    # round to its neighbour in each layer, and what it moves in the next is no larger (weights of unit variance)
    tolerance = 2 * EPS[x.dtype] * len(model.rnn_lst)
    for got, want in ((h, want_h), (c, want_c)):
        assert got.dtype == want.dtype and got.shape == want.shape and got.is_contiguous()
        error = (got.double() - want.double()).abs() / want.double().abs().clamp(min=1.0)
        assert float(error.max()) <= tolerance, float(error.max())
    return h, c


# one wavefront with work, a last wavefront with less, more steps than are in flight, projections of the same kinds, every form
SIZES = [(32, {}), (96, dict(projection_size=32)), (64, dict(bidirectional=True)), (288, dict(use_tanh=True)), (288, dict(bidirectional=True, projection_size=96)),
         (544, dict(has_skip_term=False)), (1056, dict(projection_size=544)), (2048, dict(projection_size=512)), (2048, {})]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("d,kw", SIZES)
def test_one_step(d, kw, batch, dtype):
    model = make(d, dtype, **kw)
    x = torch.randn(1, batch, model.output_size, device="cuda").to(dtype)
    c0 = torch.randn(3, batch, model.output_size, device="cuda").to(dtype)
    pad = torch.rand(1, batch, device="cuda") < 0.3
    check(model, x)
    check(model, x, c0, pad)
    check(model, x, c0.float())


@pytest.mark.parametrize("layers,taken", [(1, False), (2, True), (16, True), (17, False)])
def test_numbers_of_layers(layers, taken):
    model = make(256, torch.bfloat16, layers)
    x = torch.randn(1, 5, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        assert (model._whole_stack(x, None, None) is not None) == taken
    if taken:
        check(model, x)


def test_nans_and_the_pattern_that_stands_for_nothing():
    """A NaN, among them one whose bits are those of a word that was not written yet, stays in its row."""
    model = make(128, torch.bfloat16)
    x = torch.randn(1, 20, 128, device="cuda").to(torch.bfloat16)
    bits = x.view(torch.int16)
    bits[0, 3, 10:20] = -1
    x[0, 7, 5] = float("nan")
    x[0, 9, 6] = float("inf")
    with torch.no_grad():
        h, c = model(x)
        want_h, want_c = one_by_one(model, x)
    for got, want in ((h, want_h), (c, want_c)):
        assert torch.equal(got.isnan(), want.isnan())
        rows = [r for r in range(20) if r not in (3, 7, 9)]
        assert bool(got[:, rows].isfinite().all())
    assert bool(h[0, 3].isnan().all()) and bool(h[0, 7].isnan().all())


def test_streams_and_threads():
    models = [make(512, torch.bfloat16, 8, projection_size=128), make(320, torch.float16, 6)]
    inputs = [torch.randn(1, 16, m.output_size, device="cuda").to(m.rnn_lst[0].weight.dtype) for m in models]
    with torch.no_grad():
        want = [m(x) for m, x in zip(models, inputs)]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.no_grad(), torch.cuda.stream(stream):
            for _ in range(50):
                h, c = models[i % 2](inputs[i % 2])
                if not (torch.equal(h, want[i % 2][0]) and torch.equal(c, want[i % 2][1])):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong


def test_recorded_and_replayed():
    model = make(256, torch.bfloat16, 4, projection_size=64)
    x = torch.randn(1, 16, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        model(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            h, c = model(x)
        for _ in range(5):
            x.copy_(torch.randn(1, 16, 256, device="cuda"))
            graph.replay()
            want_h, want_c = model(x.clone())
            assert torch.equal(h, want_h) and torch.equal(c, want_c)
            torch.cuda.synchronize()


def test_layers_that_could_tell_are_called():
    x = torch.randn(1, 4, 64, device="cuda").to(torch.bfloat16)
    whole = lambda m: m._whole_stack(x, None, None) is not None

    class Own(modules.SRUCell):
        pass

    with torch.no_grad():
        assert whole(make(64, torch.bfloat16))
        calls = []
        model = make(64, torch.bfloat16)
        model.rnn_lst[1].register_forward_hook(lambda *a: calls.append(1))
        assert not whole(model)
        model(x)
        assert calls == [1]
        model = make(64, torch.bfloat16)
        model.rnn_lst[1].compute_U = lambda t: t
        assert not whole(model)
        model = make(64, torch.bfloat16)
        model.rnn_lst[1].__class__ = Own
        assert not whole(model)
        model = make(64, torch.bfloat16, dropout=0.5).train()
        assert not whole(model)
        assert whole(model.eval())
        model = make(64, torch.bfloat16)
        model.rnn_lst[1].weight = torch.nn.Parameter(model.rnn_lst[1].weight.t().contiguous().t())
        assert not whole(model) and model(x)[0].shape == x.shape
        handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
        assert not whole(make(64, torch.bfloat16))
        handle.remove()
        for other in (x.expand(2, 4, 64).contiguous(), x[..., :32], x.float()):
            assert make(64, torch.bfloat16)._whole_stack(other, None, None) is None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not whole(make(64, torch.bfloat16))
    assert not whole(make(64, torch.bfloat16))   # gradients
