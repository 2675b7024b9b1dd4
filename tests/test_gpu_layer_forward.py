"""Layers whose dense products and recurrence run in one kernel (sru_amd_layer_forward), against the
same layer in float64."""
import pytest
import torch

from sru_amd import SRUCell
from sru_amd import functional, modules

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def reference(cell, x, c0, pad):
    """The layer in float64; only what the layer itself holds in 16 bits (the projected input) is rounded."""
    L, B = x.shape[:2]
    D, d, k = cell.output_size, cell.hidden_size, cell.num_matrices
    y = x.double().reshape(L * B, -1)
    if cell.weight_proj is not None:
        y = (y @ cell.weight_proj.double()).to(x.dtype).double()
    u = (y @ cell.weight.double()).view(L, B, D, k)
    wc, bias = cell.weight_c.double(), cell.bias.double()
    scale = cell.scale_x.double() if cell.rescale else 1.0
    skip = u[..., 3] if k == 4 else x.double() * scale if cell.has_skip_term else torch.zeros_like(u[..., 0])
    h, last = torch.empty(L, B, D, dtype=torch.float64, device="cuda"), []
    for i in range(D // d):
        s = slice(i * d, (i + 1) * d)
        c = torch.zeros(B, d, dtype=torch.float64, device="cuda") if c0 is None else c0[:, s].double()
        for t in (range(L - 1, -1, -1) if i else range(L)):
            u0, u1, u2 = (u[t, :, s, n] for n in range(3))
            g1 = torch.sigmoid(u1 + wc[:D][s] * c + bias[:D][s])
            g2 = torch.sigmoid(u2 + wc[D:][s] * c + bias[D:][s])
            new = (c - u0) * g1 + u0
            out = ((torch.tanh(new) if cell.activation_type else new) - skip[t, :, s]) * g2 + skip[t, :, s]
            keep = torch.zeros(B, 1, dtype=torch.bool, device="cuda") if pad is None else pad[t][:, None]
            h[t, :, s] = torch.where(keep, torch.zeros_like(out), out)
            c = torch.where(keep, c, new)
        last.append(c)
    return h, torch.cat(last, -1)


def check(cell, x, c0, pad, route_expected=True):
    taken = []
    original = modules.layer_forward
    try:
        modules.layer_forward = lambda *a: taken.append(original(*a)) or taken[-1]
        with torch.no_grad():
            h, c = cell(x, c0, mask_pad=pad)
    finally:
        modules.layer_forward = original
    assert (taken[0] is not None) == route_expected
    want_h, want_c = reference(cell, x, c0, pad)
    # the results' own rounding, plus a flip of the last bit of a projected value here and there,
    # plus float arithmetic: two units in the last place of a value around the row's scale
    eps = 2 * EPS[x.dtype]
    for got, want in ((h, want_h), (c, want_c)):
        assert got.dtype == x.dtype
        err = (got.double() - want).abs() / want.abs().clamp(min=1.0)
        assert float(err.max()) <= eps, float(err.max())
    return h, c


def make(inp, d, dtype, **kw):
    torch.manual_seed(inp + d)
    cell = SRUCell(inp, d, rescale=True, highway_bias=-0.5, **kw).cuda().to(dtype).eval()
    with torch.no_grad():
        cell.bias += 0.3 * torch.randn_like(cell.bias)
    return cell


STEP = [(64, 64, {}), (64, 64, dict(bidirectional=True)), (96, 32, dict(n_proj=32)), (256, 256, dict(n_proj=64)),
        (288, 288, dict(use_tanh=True)), (128, 128, dict(has_skip_term=False)), (2048, 2048, dict(n_proj=512)),
        (2048, 96, {}),
        # the inner sizes where the number of steps in flight changes (512 with the recurrence, 1024 without)
        (512, 512, {}), (544, 544, {}), (512, 512, dict(has_skip_term=False)), (544, 544, dict(has_skip_term=False)),
        (1024, 96, dict(n_proj=32)), (1056, 96, dict(n_proj=64))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("inp,d,kw", STEP)
def test_one_step(inp, d, kw, batch, dtype):
    cell = make(inp, d, dtype, **kw)
    x = torch.randn(1, batch, inp, device="cuda").to(dtype)
    c0 = torch.randn(batch, cell.output_size, device="cuda").to(dtype)
    pad = torch.rand(1, batch, device="cuda") < 0.3
    check(cell, x, c0, None)
    check(cell, x, None, pad)
    check(cell, x, c0.float(), pad)


# (input, hidden, batch, length): partial groups of batch elements and of cells, an inner size at, between
# and above the register classes, a last tile of every remainder; up to 65536 columns tiles have four
# steps, above two
LONG = [(64, 64, 385, 257, dict(bidirectional=True)), (128, 64, 386, 258, dict(bidirectional=True)),
        (160, 72, 683, 259, {}), (256, 256, 131, 257, dict(bidirectional=True)), (512, 256, 128, 256, dict(bidirectional=True)),
        (512, 256, 133, 258, dict(bidirectional=True)), (288, 144, 171, 260, dict(bidirectional=True)),
        (128, 128, 384, 256, dict(n_proj=32))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("inp,d,batch,length,kw", LONG)
def test_long_sequences(inp, d, batch, length, kw, dtype):
    cell = make(inp, d, dtype, **kw)
    x = torch.randn(length, batch, inp, device="cuda").to(dtype)
    c0 = torch.randn(batch, cell.output_size, device="cuda").to(dtype)
    lens = torch.randint(1, length + 1, (batch,), device="cuda")
    pad = torch.arange(length, device="cuda")[:, None] >= lens[None, :]
    check(cell, x, c0, None)
    check(cell, x, None, pad)
    check(cell, x, c0.float(), pad)


def test_long_sequences_outside_the_route():
    big = dict(bidirectional=True)
    for inp, d, batch, length, kw in [(64, 64, 383, 256, big), (64, 64, 384, 255, big), (64, 68, 1024, 256, {}), (72, 64, 1024, 256, {}),
                                      (288, 64, 1024, 256, {}), (256, 256, 256, 256, dict(use_tanh=True)),
                                      (256, 256, 256, 256, dict(has_skip_term=False))]:
        k = 3 if not kw.get("has_skip_term", True) or inp == d * (1 + kw.get("bidirectional", False)) else 4
        plan = functional._layer_plan(torch.float16, 3, length, batch, inp, 0, d, 2 if "bidirectional" in kw else 1, k,
                                      kw.get("has_skip_term", True), int(kw.get("use_tanh", False)))
        assert plan[1] == 0


def test_one_step_outside_the_route():
    cell = make(64, 64, torch.bfloat16)
    check(cell, torch.randn(1, 65, 64, device="cuda").bfloat16(), None, None, route_expected=False)   # too many rows
    check(make(64, 40, torch.bfloat16), torch.randn(1, 4, 64, device="cuda").bfloat16(), None, None, route_expected=False)
    x = torch.randn(1, 4, 64, device="cuda").bfloat16()
    with torch.no_grad():
        two_dim = cell(x[0])
    assert two_dim[0].shape == (4, 64)
    assert torch.equal(two_dim[0], check(cell, x, None, None)[0][0])
