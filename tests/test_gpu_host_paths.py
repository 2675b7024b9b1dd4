"""The native host side (csrc/host.cpp) against the general one in functional.py: the same kernels with the
same arguments, so the same bits, over the forms of tensors that a call may come with."""
import pytest
import torch

from sru_amd import ElementwiseRecurrence, _lib, elementwise_recurrence_forward

pytestmark = pytest.mark.gpu


class General:
    """Stands for the native module where nothing is plain."""
    scan_forward = scan_backward = layer_forward = staticmethod(lambda *a: None)


class Counting:
    def __init__(self, module):
        self.module, self.plain = module, []

    def __getattr__(self, name):
        def call(*a):
            out = getattr(self.module, name)(*a)
            self.plain.append(out is not None)
            return out
        return call


def tensors(k, dtype, x_dtype, L=11, B=5, d=34, seed=0):
    g = torch.Generator().manual_seed(seed)
    D = 2 * d
    r = lambda *s: torch.randn(*s, generator=g).cuda()
    return dict(u=r(L, B, D * k).to(dtype), x=r(L, B, D).to(x_dtype), weight_c=r(2 * D), bias=r(2 * D), init=r(B, D),
                scale=torch.tensor([1.7]).cuda(), mask_c=r(B, D), mask_pad=torch.rand(L, B, generator=g).cuda() < 0.3, d=d,
                grad_h=r(L, B, D).to(dtype), grad_last=r(B, D).to(dtype))


# name -> (change to the tensors, whether the native side takes forward / backward)
FORMS = {
    "plain": (lambda t: None, True, True),
    "no options": (lambda t: t.update(init=None, scale=None, mask_c=None, mask_pad=None), True, True),
    "strided u": (lambda t: t.update(u=t["u"].transpose(0, 1).contiguous().transpose(0, 1)), False, None),
    "misaligned u": (lambda t: t.update(u=torch.cat([t["u"].flatten()[:1], t["u"].flatten()])[1:].view(t["u"].shape)), False, None),
    "strided init": (lambda t: t.update(init=t["init"].t().contiguous().t()), False, None),
    "byte mask": (lambda t: t.update(mask_pad=t["mask_pad"].to(torch.uint8)), False, None),
    "double bias": (lambda t: t.update(bias=t["bias"].double()), False, None),
    "two scales": (lambda t: t.update(scale=torch.tensor([1.7, 2.0]).cuda()), False, None),
    "strided grad_h": (lambda t: t.update(grad_h=t["grad_h"].transpose(0, 1).contiguous().transpose(0, 1)), True, False),
    "expanded grad_h": (lambda t: t.update(grad_h=t["grad_h"][:1, :1, :1].expand_as(t["grad_h"])), True, False),
    "no grad_h": (lambda t: t.update(grad_h=None), True, False),
    "no grad_last": (lambda t: t.update(grad_last=None), True, True),
}
STREAMS = [(3, torch.float32, torch.float32, True), (3, torch.bfloat16, torch.bfloat16, True), (3, torch.bfloat16, torch.float32, True),
           (4, torch.float16, torch.float16, True), (3, torch.float16, torch.float16, False)]


def one_pass(t, has_skip, hooks=None):
    leaves = {n: t[n].detach().requires_grad_() for n in ("u", "x", "weight_c", "bias", "init") if t[n] is not None}
    with hooks or torch.enable_grad():
        h, last = ElementwiseRecurrence.apply(leaves["u"], leaves["x"], leaves["weight_c"], leaves["bias"], leaves.get("init"), 0,
                                              t["d"], True, has_skip, t["scale"], t["mask_c"], t["mask_pad"])
    outs = [(o, g) for o, g in ((h, t["grad_h"]), (last, t["grad_last"])) if g is not None]
    grads = torch.autograd.grad([o for o, _ in outs], list(leaves.values()), [g for _, g in outs], allow_unused=True)
    with torch.no_grad():
        h2, last2, _ = elementwise_recurrence_forward(t["u"], t["x"], t["weight_c"], t["bias"], t["init"], 0, t["d"], True, has_skip,
                                                      t["scale"], t["mask_c"], t["mask_pad"], keep_c=False)
    return [h.detach(), last.detach(), *grads, h2, last2]


def same(a, b):
    for p, q in zip(a, b):
        assert (p is None) == (q is None)
        assert p is None or (p.dtype == q.dtype and p.shape == q.shape and torch.equal(p, q))


@pytest.mark.parametrize("k,dtype,x_dtype,has_skip", STREAMS)
@pytest.mark.parametrize("form", list(FORMS))
def test_same_bits(form, k, dtype, x_dtype, has_skip, monkeypatch):
    t = tensors(k, dtype, x_dtype)
    change, forward, backward = FORMS[form]
    change(t)
    native = Counting(_lib.host())
    monkeypatch.setattr(_lib, "host", lambda: native)
    got = one_pass(t, has_skip)
    calls = native.plain
    if form != "two scales" or (k == 3 and has_skip):     # (without a skip term from x no scale is read)
        assert calls[0] == forward and calls[-1] == forward and (backward is None or form == "no grad_h" or calls[1] == backward)
    monkeypatch.setattr(_lib, "host", lambda: General)
    same(got, one_pass(t, has_skip))


@pytest.mark.parametrize("k,dtype,x_dtype,has_skip", STREAMS)
def test_saved_tensor_hooks(k, dtype, x_dtype, has_skip):
    t = tensors(k, dtype, x_dtype)
    want = one_pass(t, has_skip)
    same(want, one_pass(t, has_skip, torch.autograd.graph.save_on_cpu()))
    # a hook that gives tensors back with other strides
    back = lambda v: v.transpose(0, -1).contiguous().transpose(0, -1) if v.dim() > 1 else v
    same(want, one_pass(t, has_skip, torch.autograd.graph.saved_tensors_hooks(lambda v: v.clone(), back)))


def test_refusals_stay():
    t = tensors(3, torch.float32, torch.float32)
    call = lambda **kw: ElementwiseRecurrence.apply(*[dict(t, **kw)[n] for n in ("u", "x", "weight_c", "bias", "init")], 0, t["d"], True,
                                                    True, t["scale"], t["mask_c"], dict(t, **kw)["mask_pad"])
    with pytest.raises(AssertionError):
        call(mask_pad=t["mask_pad"][:-1])
    with pytest.raises(ValueError):
        call(bias=t["bias"][:-1])
    with pytest.raises(ValueError):
        call(u=t["u"][:-1])
    with pytest.raises(RuntimeError):
        call(u=t["u"].cpu())
