"""The dense product of short sequences and prompts (csrc/product.hip): by itself against float64, and in
layers without gradients against the same layer as library products and recurrence."""
import ctypes

import pytest
import torch

from sru_amd import SRU, SRUCell, _lib, modules
from tests.test_abi_host import _lib_status

pytestmark = pytest.mark.gpu

CODE = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}
# half a unit in the last place of the results, relative
HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
# (rows, inner, cols): each tile at its edges and between them, inner sizes with and without a remainder, down to one
# piece, fewer tiles of them than are in flight and many more, halves of them uneven and empty
SIZES = [(1, 8, 4), (31, 24, 36), (33, 64, 100), (65, 72, 132), (7, 1032, 36), (130, 520, 68), (40, 1088, 64),
         (160, 200, 2500), (97, 264, 3204), (513, 256, 1404), (705, 264, 1092), (96, 1096, 4100), (1600, 136, 2052), (64, 3000, 64)]


# those of SIZES that float has no kernel for: few inner indices or columns, or many inner indices for the result's width
NO_FLOAT = [(1, 8, 4), (31, 24, 36), (7, 1032, 36), (130, 520, 68), (40, 1088, 64), (96, 1096, 4100), (64, 3000, 64)]


@pytest.mark.parametrize("dtype", list(CODE))
@pytest.mark.parametrize("rows,inner,cols", SIZES)
def test_product(rows, inner, cols, dtype):
    lib = _lib.load()
    g = torch.Generator().manual_seed(rows)
    x, w = torch.randn(rows, inner, generator=g).to(dtype), torch.randn(inner, cols, generator=g).to(dtype)
    out = torch.full((rows + 1, cols), float("nan"), device="cuda", dtype=dtype)   # (a row behind it, to stay as it is)
    xd, wd = x.cuda(), w.cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.sru_amd_product(CODE[dtype], rows, inner, cols, p(xd), p(wd), p(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if dtype == torch.float32 and (rows, inner, cols) in NO_FLOAT:
        assert lib.sru_amd_status_string(rc) == lib.sru_amd_status_string(_lib_status("BAD_SHAPE")) and torch.isnan(out).all()
        return
    assert rc == 0
    got = out.cpu()
    assert torch.isnan(got[rows]).all()
    want = x.double() @ w.double()
    # float sums of `inner` terms, then the result's rounding
    bound = inner * 2.0 ** -24 * (x.double().abs() @ w.double().abs()) + HALF_ULP[dtype] * want.abs() + 2.0 ** -24
    assert ((got[:rows].double() - want).abs() <= bound).all()


# (type, rows, inner, cols, rows and columns of the tile in 32, parts of the inner dimension): every kernel, cut off at its edges
TILES = [(torch.float32, 33, 72, 100, (1, 1, 1)), (torch.float32, 128, 512, 1536, (1, 1, 2)), (torch.float32, 33, 1020, 2052, (1, 1, 2)),
         (torch.float32, 705, 264, 1092, (1, 2, 1)), (torch.float32, 1601, 136, 2052, (2, 2, 1)),
         (torch.bfloat16, 31, 24, 36, (1, 1, 1)), (torch.bfloat16, 40, 1088, 68, (1, 1, 2)), (torch.bfloat16, 97, 264, 3204, (1, 2, 1)),
         (torch.float16, 62, 1544, 7684, (1, 2, 2)), (torch.bfloat16, 62, 1544, 7684, (1, 2, 2)), (torch.bfloat16, 513, 256, 1404, (2, 2, 1)),
         (torch.float16, 127, 2056, 6100, (2, 2, 2)), (torch.bfloat16, 127, 2056, 6100, (2, 2, 2)),
         (torch.bfloat16, 199, 1544, 4604, (1, 2, 1))]     # (288 tiles of 64 x 64: two rounds of smaller ones instead)


@pytest.mark.parametrize("dtype,rows,inner,cols,tile", TILES)
def test_every_tile(dtype, rows, inner, cols, tile):
    from torch.profiler import ProfilerActivity, profile
    lib = _lib.load()
    g = torch.Generator().manual_seed(rows)
    x, w = torch.randn(rows, inner, generator=g).to(dtype), torch.randn(inner, cols, generator=g).to(dtype)
    out, xd, wd = torch.full((rows + 1, cols), float("nan"), device="cuda", dtype=dtype), x.cuda(), w.cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        assert lib.sru_amd_product(CODE[dtype], rows, inner, cols, p(xd), p(wd), p(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
    name = {torch.float32: "float", torch.float16: "sru_amd::half_bits", torch.bfloat16: "sru_amd::bf16_bits"}[dtype]
    kernels = [e.name for e in seen.events() if "product_tile<" in e.name]
    assert len(kernels) == 1 and "product_tile<%s, %d, %d, %d>" % (name, *tile) in kernels[0]
    got = out.cpu()
    assert torch.isnan(got[rows]).all()
    want = x.double() @ w.double()
    bound = inner * 2.0 ** -24 * (x.double().abs() @ w.double().abs()) + HALF_ULP[dtype] * want.abs() + 2.0 ** -24   # (as above)
    assert ((got[:rows].double() - want).abs() <= bound).all()


def test_infinities_and_nan_stay_in_their_rows_and_columns():
    x, w = torch.randn(70, 72, device="cuda"), torch.randn(72, 72, device="cuda")
    x[3, 71], x[5, 0], w[7, 9] = float("inf"), float("nan"), float("-inf")
    out = torch.empty(70, 72, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert _lib.load().sru_amd_product(_lib.F32, 70, 72, 72, p(x), p(w), p(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    out, want = out.cpu(), x.cpu().double() @ w.cpu().double()
    assert torch.equal(torch.isnan(out), torch.isnan(want)) and torch.equal(torch.isinf(out), torch.isinf(want))


def both(model, *args, **kw):
    """As the kernels make it, and as library products and recurrence."""
    taken, layer, dense, host = [], modules.layer_forward, modules.dense, _lib.host().product
    spy = lambda f: lambda *a: taken.append(f(*a)) or taken[-1]
    short = args[0].dtype == torch.float32
    with torch.no_grad(), pytest.MonkeyPatch.context() as patch:
        if short:
            patch.setattr(_lib.host(), "product", spy(host))
        else:
            patch.setattr(modules, "layer_forward", spy(layer))
        got = model(*args, **kw)
        patch.setattr(modules, "layer_forward", lambda *a: None)
        patch.setattr(modules, "dense", lambda x, w: x.mm(w))
        want = model(*args, **kw)
    assert any(t is not None for t in taken) and (short or all(t is not None for t in taken))   # (a float product may be the library's)
    return got, want


# (length, batch, input, hidden, options of the stack)
LAYERS = [(20, 32, 128, 128, {}), (9, 5, 200, 200, dict(bidirectional=True)), (1, 3, 64, 64, {}), (33, 7, 96, 128, dict(projection_size=64)),
          (128, 1, 256, 256, dict(projection_size=64)), (17, 4, 96, 72, dict(layer_norm=True, rescale=True, has_skip_term=False)),
          (300, 2, 1024, 1024, dict(projection_size=256))]


@pytest.mark.parametrize("dtype", list(CODE))
@pytest.mark.parametrize("length,batch,inp,d,kw", LAYERS)
def test_layers(length, batch, inp, d, kw, dtype):
    if length == 1 and dtype != torch.float32:
        pytest.skip("one step in 16 bits has kernels of its own")
    torch.manual_seed(d)
    model = SRU(inp, d, num_layers=2, highway_bias=-1.0, **kw).cuda().to(dtype).eval()
    x = torch.randn(length, batch, inp, device="cuda").to(dtype)
    c0 = torch.randn(2, batch, model.output_size, device="cuda").to(dtype)
    pad = torch.rand(length, batch, device="cuda") < 0.3
    for args in ((x,), (x, c0, pad)):
        (h, c), (h2, c2) = both(model, *args[:2], mask_pad=args[2] if len(args) > 2 else None)
        for a, b in ((h, h2), (c, c2)):
            assert a.dtype == b.dtype == dtype and a.shape == b.shape
            # values of order one from two layers: sums of up to 1024 terms in another order, and in 16 bits a
            # result's last bit flipped here and there, which the state carries on
            tol = 1e-4 if dtype == torch.float32 else 8 * HALF_ULP[dtype]
            assert float(((a.double() - b.double()).abs() / b.double().abs().clamp(min=1.0)).max()) <= tol


def test_layer_in_a_graph():
    model = SRU(128, 128, num_layers=2).cuda().eval()
    x = torch.randn(20, 32, 128, device="cuda")
    with torch.no_grad():
        model(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(x)
        for _ in range(4):
            x.copy_(torch.randn_like(x))
            graph.replay()
            replayed = [o.clone() for o in out]
            want = model(x)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(replayed, want))


def test_forms_that_go_the_general_way():
    """Strided, misaligned or mixed tensors give what they gave, and what was refused stays refused."""
    cell = SRUCell(64, 64).cuda().eval()
    x = torch.randn(6, 5, 64, device="cuda")
    with torch.no_grad():
        want = cell(x)
        strided = x.transpose(0, 1).contiguous().transpose(0, 1)
        shifted = torch.cat([x.flatten()[:1], x.flatten()])[1:].view(x.shape)
        for other in (strided, shifted):
            for a, b in zip(cell(other), want):
                assert torch.allclose(a, b, rtol=1e-5, atol=1e-5)
        with pytest.raises(Exception):
            cell(x, torch.randn(5, 63, device="cuda"))
        with pytest.raises(Exception):
            cell(x.bfloat16())
