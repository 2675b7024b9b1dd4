"""Whole stacks in one launch (sru_amd_stack_forward), one time step or a short sequence, against the same layers called one by
one, which test_gpu_layer_forward.py holds against float64."""
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


# more pieces than workgroups: the least number of them, three layers' worth, 128, two layers' with a projection, all the chip
@pytest.mark.parametrize("d,layers,kw", [(128, 16, {}), (576, 6, {}), (1600, 4, {}), (1024, 5, dict(projection_size=256)), (2048, 5, dict(projection_size=512)),
                                         (2048, 4, dict(projection_size=1792))])
def test_pieces_beyond_the_workgroups(d, layers, kw):
    model = make(d, torch.bfloat16, layers, **kw)
    for batch in (1, 20):
        check(model, torch.randn(1, batch, d, device="cuda").to(torch.bfloat16))


# sequences: chunks of 32 rows and of 64, one chunk and fewer of them than lie between two layers, a last chunk of few steps, a
# second half of rows that is not there, a last group of 32 cells, one row to four, rows that do not divide a chunk, inner
# sizes below, at and past what passes through LDS at once, the fewest layers and the most (of some width: sixteen layers of 32
# cells make a single rounding grow until the two errors compared below differ by chance, 0.5 to 10 over 16 inputs, 0.95 on average)
SEQUENCES = [(32, 1, 64, {}), (64, 1, 32, {}), (64, 1, 256, dict(layers=16)), (65, 1, 96, dict(projection_size=32)), (100, 2, 64, dict(use_tanh=True)), (257, 1, 288, {}),
             (300, 1, 544, dict(projection_size=96)), (289, 1, 512, dict(has_skip_term=False)), (290, 1, 544, {}), (129, 2, 480, dict(layers=6)),
             (130, 4, 128, dict(layers=5, projection_size=32)), (200, 3, 256, dict(layers=6, projection_size=64)), (64, 3, 64, {}),
             (100, 1, 2048, dict(layers=10, projection_size=512)), (513, 1, 2048, dict(layers=6, projection_size=512)),
             (700, 1, 1280, dict(layers=10, projection_size=544)), (500, 3, 320, dict(layers=10)), (491, 1, 1024, dict(layers=6))]

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("length,batch,d,kw", SEQUENCES)
def test_sequences(length, batch, d, kw, dtype):
    model = make(d, dtype, **kw)
    x = torch.randn(length, batch, d, device="cuda").to(dtype)
    c0 = torch.randn(len(model.rnn_lst), batch, d, device="cuda").to(dtype)
    pad = torch.rand(length, batch, device="cuda") < 0.3
    pad[-3:] = True
    with torch.no_grad():
        for state, mask in ((None, None), (c0, pad), (c0.float(), None)):
            assert model._whole_stack(x, state, mask) is not None
            got, want = model(x, state, mask_pad=mask), one_by_one(model, x, state, mask_pad=mask)
            wide = model.float()(x.float(), None if state is None else state.float(), mask_pad=mask)
            model.to(dtype)
            for a, b, exact in zip(got, want, wide):
                # U stays in float here and is rounded on the way to the recurrence there: no further from the result in
                # float throughout, of which both are a few roundings of 16 bits per layer away (the norm of N independent
                # errors varies by 1 / sqrt(2 N); the state carries one over some four steps, so of two norms' ratio
                # three deviations are 6 / sqrt(numel))
                exact, norm = exact.double(), exact.double().norm()
                assert float((a.double() - exact).norm() / norm) <= (1.05 + 6 / a.numel() ** 0.5) * float((b.double() - exact).norm() / norm)
                assert float((a.double() - b.double()).norm() / norm) <= 4 * EPS[dtype]
                # one wrong cell or step is nothing in a norm: no element is further off than eight times that share (the largest
                # of 10^7 normal deviates is 5.4) of the elements' mean square, or of itself where it is larger
                size = b.double().abs().clamp(min=float(norm / a.numel() ** 0.5))
                assert float(((a.double() - b.double()).abs() / size).max()) <= 32 * EPS[dtype]
                if mask is not None and a.shape[0] == length:
                    assert not bool(a[mask].any())


@pytest.mark.parametrize("length,batch,d,kw,taken", [(32, 1, 64, {}, True), (31, 1, 64, {}, False), (64, 4, 64, {}, True), (64, 5, 64, {}, False), (64, 1, 48, {}, False),
                                                    (64, 1, 544, {}, False), (256, 1, 544, {}, True), (256, 1, 1056, {}, False),
                                                    (130, 4, 128, dict(projection_size=32), False), (64, 1, 64, dict(bidirectional=True), False)])
def test_sequences_that_are_taken(length, batch, d, kw, taken):
    model = make(d, torch.bfloat16, **kw)
    with torch.no_grad():
        assert (model._whole_stack(torch.zeros(length, batch, model.output_size, device="cuda", dtype=torch.bfloat16), None, None) is not None) == taken


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


@pytest.mark.parametrize("length,batch,d,kw", [(130, 1, 256, dict(layers=4, projection_size=64)), (200, 2, 256, dict(layers=6)), (513, 1, 512, dict(layers=6, projection_size=128)),
                                              (150, 3, 128, dict(layers=8))])
def test_nans_and_infinities_in_sequences(length, batch, d, kw):
    """Over several chunks and layers, with padding and a state: they stay in their batch row, from their step on, and come out where they do layer by
    layer, whatever their bits (of a word that was not written yet, and of a NaN sum like the one that marks a padded step)."""
    model = make(d, torch.bfloat16, **kw)
    x = torch.randn(length, batch, d, device="cuda").to(torch.bfloat16)
    c0 = torch.randn(len(model.rnn_lst), batch, d, device="cuda").to(torch.bfloat16)
    pad = torch.rand(length, batch, device="cuda") < 0.2
    at = length // 2                                       # of the last batch row; the others stay finite
    pad[at - 1:at + 4, -1] = False
    cases = {"pattern": lambda x, c: x.view(torch.int16)[at, -1, 4:9].fill_(-1), "all bits": lambda x, c: x.view(torch.int16)[at, -1].fill_(-1),
             "nan": lambda x, c: x[at, -1, 3].fill_(float("nan")), "negative nan": lambda x, c: x.view(torch.int16)[at, -1, 3].fill_(-64),
             "inf": lambda x, c: x[at, -1, 7].fill_(float("inf")), "state": lambda x, c: c[0, -1, 5].fill_(float("nan")),
             "state's infinity": lambda x, c: c[1, -1, 6].fill_(float("-inf"))}
    with torch.no_grad():
        for name, plant in cases.items():
            inputs, states = x.clone(), c0.clone()
            plant(inputs, states)
            for mask in (None, pad):
                assert model._whole_stack(inputs, states, mask) is not None
                got, want = model(inputs, states, mask_pad=mask), one_by_one(model, inputs, states, mask_pad=mask)
                for a, b in zip(got, want):
                    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), name
                    assert bool(a[:, :-1].isfinite().all())
                    a, b = a[b.isfinite()].double(), b[b.isfinite()].double()
                    size = b.abs().clamp(min=float(b.square().mean().sqrt())) if b.numel() else b
                    assert not bool(((a - b).abs() > 32 * EPS[torch.bfloat16] * size).any()), name
                h = got[0]
                assert bool(h.isnan().any()) and ("state" in name or bool(h[:at].isfinite().all()))
                assert mask is None or not bool(h[mask].any())


def test_streams_and_threads():
    models = [make(512, torch.bfloat16, 8, projection_size=128), make(320, torch.float16, 6), make(256, torch.bfloat16, 5)]
    inputs = [torch.randn(length, batch, m.output_size, device="cuda").to(m.rnn_lst[0].weight.dtype) for m, length, batch in zip(models, (1, 1, 150), (16, 16, 1))]
    with torch.no_grad():
        assert all(m._whole_stack(x, None, None) is not None for m, x in zip(models, inputs))
        want = [m(x) for m, x in zip(models, inputs)]
    torch.cuda.synchronize()
    wrong, done = [], []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.no_grad(), torch.cuda.stream(stream):
            for _ in range(50):
                h, c = models[i % 3](inputs[i % 3])
                if not (torch.equal(h, want[i % 3][0]) and torch.equal(c, want[i % 3][1])):
                    wrong.append(i)
                done.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong and len(done) == 6 * 50


def test_no_room_for_the_workspace():
    """Where the allocator refuses it, the layers are called one by one, which hold less at a time."""
    model = make(2048, torch.bfloat16, 10, projection_size=512)
    x = torch.randn(1024, 1, 2048, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        want = one_by_one(model, x)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        room = 1024 * (10 * 512 + 9 * 2048) * 2     # of the workspace, at the least
        held, before = [], torch.cuda.memory_reserved()
        while torch.cuda.memory_reserved() == before:    # what earlier tests left in the allocator's segments
            held.append(torch.empty(room, dtype=torch.uint8, device="cuda"))
        held.pop()
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_reserved()
        one_by_one(model, x)
        growth = torch.cuda.max_memory_reserved() - before
        torch.cuda.empty_cache()
        assert growth < room
        torch.cuda.set_per_process_memory_fraction((before + growth + (2 << 20)) / torch.cuda.get_device_properties(0).total_memory)
        try:
            got = model(x)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        assert model._whole_stack(x, None, None) is not None


@pytest.mark.parametrize("replace", ["parameter", "memory"])
@pytest.mark.parametrize("length", [1, 130])
def test_weights_replaced_by_another_thread(length, replace):
    """A call reads the weights that it found: they are equal ones here, and what is freed meanwhile becomes NaNs (all on one
    stream, in the order of the calls)."""
    model = make(256, torch.bfloat16, 8, projection_size=64)
    x = torch.randn(length, 1, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        assert model._whole_stack(x, None, None) is not None
        want = model(x)
    done, failed, rounds = threading.Event(), [], 0

    def work():
        try:
            while not done.is_set():
                for cell in model.rnn_lst:
                    for name in ("weight", "weight_proj", "weight_c", "bias"):
                        old = getattr(cell, name)
                        size, new = old.shape, old.detach().clone()
                        if replace == "memory":
                            old.data = new
                        else:
                            setattr(cell, name, torch.nn.Parameter(new))
                        del old, new
                        torch.full(size, float("nan"), device="cuda", dtype=torch.bfloat16)
        except BaseException as e:
            failed.append(e)

    thread = threading.Thread(target=work)
    thread.start()
    try:
        with torch.no_grad():
            for rounds in range(1, 301):
                got = model(x)
                if not all(torch.equal(a, b) for a, b in zip(got, want)):
                    failed.append(rounds)
                    break
    finally:
        done.set()
        thread.join()
    assert not failed and rounds == 300


@pytest.mark.parametrize("length,batch", [(1, 16), (130, 1)])
def test_recorded_and_replayed(length, batch):
    model = make(256, torch.bfloat16, 4, projection_size=64)
    x = torch.randn(length, batch, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        model(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            assert model._whole_stack(x, None, None) is not None
            h, c = model(x)
        for _ in range(5):
            x.copy_(torch.randn(length, batch, 256, device="cuda"))
            graph.replay()
            want_h, want_c = model(x.clone())
            assert torch.equal(h, want_h) and torch.equal(c, want_c)
            for got, want in zip((h, c), one_by_one(model, x)):    # (and not both of them stale: as in test_sequences)
                assert float((got.double() - want.double()).norm() / want.double().norm()) <= 4 * EPS[torch.bfloat16]
            torch.cuda.synchronize()


@pytest.mark.parametrize("d,layers,rows,taken", [(64, 2, 16, False), (32, 3, 48, False), (256, 8, 16, True)])
def test_one_step_in_a_graph_where_launches_cost_the_host_nothing(d, layers, rows, taken):
    model = make(d, torch.bfloat16, layers)
    x = torch.randn(1, rows, d, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        assert model._whole_stack(x, None, None) is not None
        one_by_one(model, x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            assert (model._whole_stack(x, None, None) is not None) == taken
            h, c = model(x)
        for _ in range(3):
            x.copy_(torch.randn(1, rows, d, device="cuda"))
            graph.replay()
            for want in (one_by_one(model, x), model(x)):   # (the same sums, up to a contraction: see check)
                for a, b in zip((h, c), want):
                    assert float(((a.double() - b.double()).abs() / b.double().abs().clamp(min=1.0)).max()) <= 2 * EPS[torch.bfloat16] * layers
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
