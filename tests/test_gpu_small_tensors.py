"""Small tensors held in the 16-bit stream type: every kernel decodes them as it reads them, so the
results are bit for bit those of float copies of the same values."""
import pytest
import torch

from sru_amd import ElementwiseRecurrence, elementwise_recurrence_forward

pytestmark = pytest.mark.gpu

# (L, B, d, dirs, k): lane pairs, paired lanes with a partial wavefront, two columns per lane,
# the general kernels (odd width), one step
SHAPES = [(19, 3, 64, 2, 3), (17, 5, 50, 2, 4), (9, 130, 512, 2, 3), (11, 3, 33, 1, 3), (1, 16, 64, 1, 3)]


def _inputs(L, B, d, dirs, k, dtype):
    gen = torch.Generator("cuda").manual_seed(L * 1000 + d)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    D = d * dirs
    mask_c = (torch.rand(B, D, generator=gen, device="cuda") < 0.8).to(dtype) / 0.75
    pad = torch.rand(L, B, generator=gen, device="cuda") < 0.2
    return dict(u=r(L, B, D * k), x=r(L, B, D), weight_c=r(2 * D), bias=r(2 * D), init=r(B, D),
                scale_x=torch.full((1,), 1.7, device="cuda", dtype=dtype), mask_c=mask_c, mask_pad=pad)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("keep_c", [False, True])
def test_forward_reads_16_bit_small_tensors(shape, dtype, keep_c):
    L, B, d, dirs, k = shape
    t = _inputs(*shape, dtype)
    run = lambda **o: elementwise_recurrence_forward(
        activation_type=0, d_out=d, bidirectional=dirs == 2, has_skip_term=True, keep_c=keep_c, **dict(t, **o))
    want = run(**{n: t[n].float() for n in ("weight_c", "bias", "init", "scale_x", "mask_c")})
    for names in (("weight_c", "bias", "init", "scale_x", "mask_c"), ("bias",), ("init", "mask_c")):
        got = run(**{n: t[n].float() for n in ("weight_c", "bias", "init", "scale_x", "mask_c") if n not in names})
        for a, b in zip(want, got):
            assert (a is None and b is None) or (a.dtype == b.dtype and torch.equal(a, b)), names


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
def test_backward_reads_a_16_bit_gradient_of_the_last_state(shape, dtype):
    L, B, d, dirs, k = shape
    t = _inputs(*shape, dtype)
    u, x = t["u"].requires_grad_(), t["x"].requires_grad_(k == 3)
    wc, bias, init = (t[n].float().requires_grad_() for n in ("weight_c", "bias", "init"))
    h, last = ElementwiseRecurrence.apply(u, x, wc, bias, init, 0, d, dirs == 2, True, t["scale_x"], t["mask_c"],
                                          t["mask_pad"])
    assert last.dtype == dtype
    gl = torch.randn(B, d * dirs, device="cuda").to(dtype)
    inputs = [u, wc, bias, init] + ([x] if k == 3 else [])
    got = torch.autograd.grad([last], inputs, [gl], retain_graph=True)
    want = torch.autograd.grad([last.float()], inputs, [gl.float()])    # arrives as dtype again, through a cast
    for a, b in zip(want, got):
        assert torch.equal(a, b)
    # one step: the gradient of the initial state written out
    if L == 1:
        live = ~t["mask_pad"][0]
        g1 = torch.sigmoid(u.float().view(B, -1, k)[..., 1] + wc[:d * dirs] * init + bias[:d * dirs])
        expect = torch.autograd.grad(torch.where(live[:, None], (init - u.float().view(B, -1, k)[..., 0]) * g1, init),
                                     init, gl.float(), retain_graph=False)[0]
        assert torch.allclose(got[3], expect, rtol=2e-6, atol=2e-6)
