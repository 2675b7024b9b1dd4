"""CPU-only checks of the boundary: the library loads, exports every symbol the header
declares, and rejects bad arguments before anything reaches a GPU."""
import ctypes
import os
import re

import pytest

from sru_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "sru_amd.h")).read()
    code = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(sru_amd_[a-z_]+)\s*\(", code))
    assert declared == set(_lib.SIGNATURES), (declared, set(_lib.SIGNATURES))
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name), name
    assert _lib.load().sru_amd_abi_version() == int(re.search(r"SRU_AMD_ABI_VERSION\s+(\d+)", header).group(1))


def test_struct_layout_matches_header():
    assert ctypes.sizeof(_lib.Shape) == 56
    assert _lib.Shape.dirs.offset == 24 and _lib.Shape.dtype.offset == 44
    assert _lib.Shape.state_interval.offset == 48 and _lib.Shape.x_dtype.offset == 52


def _shape(**kw):
    base = dict(length=4, batch=2, hidden=8, dirs=2, k=3, activation_type=0, skip_type=1,
                is_custom=0, dtype=0, state_interval=0, x_dtype=0)
    base.update(kw)
    return _lib.Shape(*[base[f[0]] for f in _lib.Shape._fields_])


FAKE = ctypes.c_void_p(0x1000)  # never dereferenced: validation fails first


@pytest.mark.parametrize("kw,code", [
    (dict(length=0), 2), (dict(batch=-1), 2), (dict(hidden=0), 2), (dict(hidden=1 << 31), 2),
    (dict(length=1 << 60), 2), (dict(dirs=3), 3), (dict(k=5), 3), (dict(k=2), 3),
    (dict(activation_type=2), 3), (dict(skip_type=3), 3), (dict(skip_type=1, k=4), 3),
    (dict(skip_type=2, k=3), 3), (dict(is_custom=2), 3), (dict(dtype=7), 4),
    (dict(state_interval=4), 3), (dict(state_interval=8, dtype=3), 3),   # double streams: no checkpoints
    (dict(state_interval=8, is_custom=1, activation_type=1), 3), (dict(state_interval=8, skip_type=0, k=4), 3),
    (dict(state_interval=8, dtype=2, hidden=7), 3), (dict(state_interval=8, dtype=1, hidden=1), 3),
    # a float x beside 16-bit streams: plain layer only, even hidden; with float streams the field changes nothing
    (dict(x_dtype=2), 4), (dict(x_dtype=1, dtype=2, state_interval=8, is_custom=1), 3),
    (dict(x_dtype=1, dtype=1, state_interval=8, activation_type=1), 3), (dict(x_dtype=1, dtype=2, hidden=7), 3),
])
def test_forward_rejects_bad_shapes(kw, code):
    lib = _lib.load()
    s = _shape(**kw)
    assert lib.sru_amd_forward(ctypes.byref(s), *([FAKE] * 11), None) == code
    assert lib.sru_amd_backward_workspace_bytes(ctypes.byref(s)) == 0
    assert lib.sru_amd_state_bytes(ctypes.byref(s)) == 0
    assert lib.sru_amd_backward(ctypes.byref(s), *([FAKE] * 17), 1 << 20, None) == code


def test_null_and_misaligned_pointers_and_workspace():
    lib = _lib.load()
    s = _shape()
    assert lib.sru_amd_forward(None, *([FAKE] * 11), None) == 1
    args = [FAKE] * 11
    for required in (0, 1, 2, 3, 8, 10):   # u, x (skip from x), weight_c, bias, h, c_last (c_init may be NULL: zeros)
        bad = list(args)
        bad[required] = None
        assert lib.sru_amd_forward(ctypes.byref(s), *bad, None) == 1, required
    odd = ctypes.c_void_p(0x1002)
    bad = list(args)
    bad[0] = odd
    assert lib.sru_amd_forward(ctypes.byref(s), *bad, None) == 5
    s4 = _shape(k=4, skip_type=2)
    bad = list(args)
    bad[0] = ctypes.c_void_p(0x1008)            # k=4 float groups move as 16-byte vectors
    assert lib.sru_amd_forward(ctypes.byref(s4), *bad, None) == 5
    need = lib.sru_amd_backward_workspace_bytes(ctypes.byref(s))
    assert need == 4 * 4 * 2 * 16
    assert lib.sru_amd_state_bytes(ctypes.byref(s)) == 4 * 2 * 16 * 4           # (L, B, D') floats
    assert lib.sru_amd_state_bytes(ctypes.byref(_shape(dtype=2))) == 4 * 2 * 16 * 2
    assert lib.sru_amd_state_bytes(ctypes.byref(_shape(state_interval=8))) == 1 * 2 * 16 * 4
    assert lib.sru_amd_state_bytes(ctypes.byref(_shape(length=33, state_interval=8, dtype=1))) == 4 * 2 * 16 * 4
    # double streams: the state after every step in double, and double partial sums
    assert lib.sru_amd_state_bytes(ctypes.byref(_shape(dtype=3))) == 4 * 2 * 16 * 8
    assert lib.sru_amd_backward_workspace_bytes(ctypes.byref(_shape(dtype=3))) == 4 * 8 * 2 * 16
    bad = list(args)
    bad[3] = ctypes.c_void_p(0x1004)            # with double streams the small tensors are doubles too
    assert lib.sru_amd_forward(ctypes.byref(_shape(dtype=3)), *bad, None) == 5
    assert lib.sru_amd_backward(ctypes.byref(s), *([FAKE] * 16), None, need, None) == 6
    assert lib.sru_amd_backward(ctypes.byref(s), *([FAKE] * 17), need - 1, None) == 6
    # u, x, weight_c, bias, c, grad_h, grad_u, grad_x, grad_wc, grad_bias, grad_init
    # (c_init = 4 and grad_last = 10 may be NULL: zeros)
    for required in (0, 1, 2, 3, 8, 9, 11, 12, 13, 14, 15):
        bad = [FAKE] * 17                        # e.g. 12: grad_x is required when the skip term is x
        bad[required] = None
        assert lib.sru_amd_backward(ctypes.byref(s), *bad, need, None) == 1, required


def test_float_x_beside_16bit_streams_needs_checkpoints_or_no_state():
    lib = _lib.load()
    s = _shape(dtype=2, x_dtype=1, state_interval=1)
    assert lib.sru_amd_forward(ctypes.byref(s), *([FAKE] * 11), None) == 3       # c given, state after every step
    assert lib.sru_amd_backward(ctypes.byref(s), *([FAKE] * 17), 1 << 20, None) == 3
    s = _shape(dtype=2, x_dtype=1, state_interval=8)
    bad = [FAKE] * 11
    bad[1] = ctypes.c_void_p(0x1002)             # the float x must be 4-byte aligned
    assert lib.sru_amd_forward(ctypes.byref(s), *bad, None) == 5


def test_static_backward_checks_sizes_before_anything_else():
    # the allocation-free entry point refuses more columns than its built-in array holds
    lib = _lib.load()
    wide = _shape(batch=_lib.STATIC_MAX_COLUMNS // 16 + 1)
    assert lib.sru_amd_backward_static(ctypes.byref(wide), *([FAKE] * 16), None) == 8
    half = _shape(batch=_lib.STATIC_MAX_COLUMNS // 32 + 1, dtype=3)   # double partial sums: half the columns
    assert lib.sru_amd_backward_static(ctypes.byref(half), *([FAKE] * 16), None) == 8
    assert lib.sru_amd_backward_static(ctypes.byref(_shape(k=5)), *([FAKE] * 16), None) == 3
    assert lib.sru_amd_backward_static(None, *([FAKE] * 16), None) == 1


def test_layer_norm_entry_points_validate_before_launching():
    lib = _lib.load()
    f32 = 0
    fwd = lambda rows, cols, x=FAKE, dx=f32, dy=f32: lib.sru_amd_layer_norm_forward(
        rows, cols, x, dx, FAKE, FAKE, ctypes.c_float(1e-5), FAKE, dy, FAKE, FAKE, None)
    assert fwd(0, 64) == 2 and fwd(4, 0) == 2 and fwd(4, 12) == 2          # cols must be a multiple of 8
    assert fwd(4, _lib.NORM_MAX_FEATURES + 8) == 2
    assert fwd(4, 64, dx=9) == 4 and fwd(4, 64, dy=5) == 4 and fwd(4, 64, dx=3) == 4   # no double rows
    assert fwd(4, 64, x=None) == 1
    assert fwd(4, 64, x=ctypes.c_void_p(0x1004)) == 5
    need = lib.sru_amd_layer_norm_backward_workspace_bytes(4, 64)
    # one (2, cols) float row per workgroup of the backward kernel: one workgroup here, 512 at most
    assert need == 2 * 64 * 4 and lib.sru_amd_layer_norm_backward_workspace_bytes(4, 12) == 0
    assert lib.sru_amd_layer_norm_backward_workspace_bytes(16384, 2048) == 512 * 2 * 2048 * 4
    assert lib.sru_amd_layer_norm_backward_workspace_bytes(10 ** 6, 4096) == 512 * 2 * 4096 * 4   # 8 wavefronts per row
    gw = ctypes.c_void_p(0x2000)
    gb = ctypes.c_void_p(0x2000 + 64 * 4)
    bwd = lambda ws, nbytes, gbias=gb: lib.sru_amd_layer_norm_backward(
        4, 64, FAKE, f32, FAKE, FAKE, FAKE, FAKE, f32, FAKE, gw, gbias, ws, nbytes, None)
    assert bwd(None, need) == 6 and bwd(FAKE, need - 1) == 6
    assert bwd(FAKE, need, gbias=ctypes.c_void_p(0x3000)) == 5          # the two sums must be adjacent


def test_status_strings_and_python_error_mapping():
    for code in range(0, 9):
        assert _lib.status_string(code)
    with pytest.raises(ValueError):
        _lib.check(3, "x")
    with pytest.raises(RuntimeError):
        _lib.check(7, "x")


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libsru_amd.so"))
    with pytest.raises(_lib.LibraryError):
        _lib.load()


def test_function_refuses_cpu_tensors():
    import torch
    from sru_amd import ElementwiseRecurrence
    L, B, d = 3, 2, 4
    with pytest.raises(RuntimeError):
        ElementwiseRecurrence.apply(torch.randn(L, B, 3 * d), torch.randn(L, B, d), torch.randn(2 * d),
                                    torch.randn(2 * d), torch.zeros(B, d), 0, d, False, True, None)


def test_plain_c_caller_is_built_and_links_against_the_library():
    """sru_amd/serve_forward (no Python, no torch) starts, i.e. finds libsru_amd.so and the HIP
    runtime next to it, and refuses a wrong argument list before it touches any device."""
    import subprocess
    program = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sru_amd", "serve_forward")
    assert os.path.exists(program), "run python -m sru_amd.build"
    proc = subprocess.run([program], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True, timeout=60)
    assert proc.returncode == 64 and "usage:" in proc.stderr


@pytest.mark.parametrize("state", ["right", "other torch", "missing"])
def test_native_host_code_is_used_with_its_own_torch_only(state, monkeypatch):
    """Without it (not built, or built for another release of torch) calls go the general way, which
    needs the kernel library alone."""
    import sys
    import types
    import sru_amd
    import torch
    module = types.ModuleType("sru_amd._host")
    module.torch_version = torch.__version__ if state == "right" else "1.0"
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.setattr(sru_amd, "_host", module, raising=False)
    if state == "missing":
        monkeypatch.delattr(sru_amd, "_host")
    monkeypatch.setitem(sys.modules, "sru_amd._host", None if state == "missing" else module)
    if state == "right":
        assert _lib.host() is module
    else:
        with pytest.warns(RuntimeWarning, match="rebuild"):
            host = _lib.host()
        assert _lib.host() is host and host.scan_forward(1, 2) is None and host.scan_backward() is None and host.layer_forward() is False


def test_native_host_code_is_built_for_this_torch():
    import torch
    assert _lib.host().torch_version == torch.__version__


# (inner, hidden, directions, streams, batch, whether the long-sequence kernel takes it): sizes on both sides of
# a round of workgroups, of cells that fill no group of 64 and of products that fill no tile, as measured
# (512 steps, us: two calls against the kernel with the better tile)
@pytest.mark.parametrize("inner,hidden,dirs,k,batch,taken", [
    (256, 256, 2, 4, 256, True),      # 357 / 166
    (256, 256, 2, 4, 320, True),      # 477 / 301
    (512, 256, 2, 3, 256, True),      # 356 / 252
    (512, 256, 2, 3, 320, True),      # 486 / 398
    (288, 256, 2, 3, 132, False),     # 204 / 219
    (288, 256, 2, 3, 264, False),     # 353 / 392
    (288, 144, 2, 3, 171, False),     # 190 / 219
    (288, 144, 2, 3, 284, True),      # 271 / 221
    (288, 144, 2, 3, 341, False),     # 325 / 391
    (288, 144, 2, 3, 512, True),      # 491 / 392
    (160, 72, 2, 4, 512, True),       # 243 / 161
    (64, 8, 1, 4, 8192, True),        # 367 / 342
])
def test_long_sequence_route_goes_by_rounds_of_workgroups(inner, hidden, dirs, k, batch, taken):
    shape = _lib.Shape(512, batch, hidden, dirs, k, 0, 1 if k == 3 else 2, 0, _lib.F16, 1, _lib.X_AS_STREAMS)
    route = _lib.load().sru_amd_layer_route(ctypes.byref(shape), inner, 0)
    assert route == (_lib.LAYER_ROWS if taken else 0)


# (in_features, n_proj, rows, whether the one-step kernels take it), at the ends of the ranges of inner sizes
@pytest.mark.parametrize("inner,n_proj,rows,taken", [
    (3072, 0, 16, True), (3104, 0, 16, False), (2560, 0, 32, True), (2592, 0, 32, False), (3072, 0, 17, False),
    (2048, 0, 64, True), (2080, 0, 64, False), (2560, 0, 33, False), (1024, 0, 65, False),
    (4096, 1024, 16, True), (4128, 1024, 16, False), (3072, 768, 32, True), (4096, 1024, 17, False),
    (2560, 640, 64, True), (3072, 768, 33, False), (4096, 3104, 1, False), (8192, 0, 1, False)])
def test_one_step_route_ends_where_library_products_are_faster(inner, n_proj, rows, taken):
    shape = _lib.Shape(1, rows, 512, 1, 4, 0, 2, 0, _lib.BF16, 1, _lib.X_AS_STREAMS)
    assert _lib.load().sru_amd_layer_route(ctypes.byref(shape), inner, n_proj) == (_lib.LAYER_STEP if taken else 0)


@pytest.mark.parametrize("dtype,rows,inner,cols,taken", [
    (_lib.F32, 640, 128, 384, 1), (_lib.F32, 640, 126, 384, 0), (_lib.F32, 640, 128, 382, 0), (_lib.F32, 640, 60, 384, 0), (_lib.F32, 640, 128, 60, 0), (_lib.F32, 128, 1024, 2048, 1),
    (_lib.F32, 128, 1024, 2044, 0), (_lib.F32, 128, 1028, 4096, 0), (_lib.BF16, 512, 512, 6144, 1), (_lib.BF16, 512, 516, 6144, 0),
    (_lib.F16, 1, 8, 4, 1), (_lib.F16, 512, 2048, 6144, 0), (_lib.F64, 64, 64, 64, 0), (_lib.BF16, 0, 64, 64, 0), (9, 64, 64, 64, 0)])
def test_product_wanted(dtype, rows, inner, cols, taken):
    lib = _lib.load()
    assert lib.sru_amd_product_wanted(dtype, rows, inner, cols) == taken
    # (nothing is launched: null pointers, or sizes that are not taken)
    text = lib.sru_amd_status_string(lib.sru_amd_product(dtype, rows, inner, cols, None, None, None, None))
    assert text == lib.sru_amd_status_string(_lib_status("NULL_POINTER" if taken else "BAD_SHAPE"))


@pytest.mark.parametrize("dtype,rows,inner,cols,wanted", [
    (_lib.BF16, 512, 512, 6144, 1), (_lib.BF16, 1000, 256, 3500, 1), (_lib.BF16, 1001, 256, 3500, 0), (_lib.F16, 3007, 128, 3584, 0),
    (_lib.BF16, 1000, 520, 1000, 1), (_lib.BF16, 1001, 520, 1000, 0), (_lib.BF16, 777, 640, 1920, 0), (_lib.F32, 2000, 384, 1000, 1),
    (_lib.F32, 500, 500, 2400, 1), (_lib.F32, 501, 500, 2400, 0)])
def test_a_product_may_be_taken_and_not_wanted(dtype, rows, inner, cols, wanted):
    lib = _lib.load()
    assert lib.sru_amd_product_wanted(dtype, rows, inner, cols) == wanted
    assert lib.sru_amd_product(dtype, rows, inner, cols, None, None, None, None) == _lib_status("NULL_POINTER")


def _lib_status(name):
    header = open(os.path.join(ROOT, "include", "sru_amd.h")).read()
    return int(re.search(r"SRU_AMD_ERR_%s\s*=?\s*(\d+)" % name, header).group(1))


@pytest.mark.parametrize("dtype,rows,inner,cols,taken", [
    (_lib.BF16, 8192, 512, 6144, 1), (_lib.F16, 8192, 128, 384, 1), (_lib.F16, 3000, 512, 3072, 1), (_lib.F16, 4096, 256, 1024, 0), (_lib.F32, 8192, 512, 6144, 0), (_lib.BF16, 2999, 512, 6144, 0),
    (_lib.BF16, 8192, 516, 6144, 0), (_lib.BF16, 8192, 512, 1540, 0), (_lib.BF16, 8192, 1032, 3072, 0), (_lib.BF16, 8192, 128, 376, 0),
    (_lib.BF16, 1 << 20, 1024, 3072, 0), (_lib.BF16, 8192, -8, -8, 0), (_lib.BF16, 1 << 62, 1 << 62, 1 << 62, 0)])
def test_product_grad_sizes(dtype, rows, inner, cols, taken):
    lib = _lib.load()
    assert (lib.sru_amd_product_grad_workspace_bytes(dtype, rows, inner, cols) > 0) == bool(taken)
    rc = lib.sru_amd_product_grad(dtype, rows, inner, cols, FAKE, FAKE, dtype, None, None, 0, None)
    assert lib.sru_amd_status_string(rc) == lib.sru_amd_status_string(_lib_status("NULL_POINTER" if taken else "BAD_SHAPE"))
    if taken:
        assert lib.sru_amd_product_grad(dtype, rows, inner, cols, FAKE, FAKE, dtype, FAKE, None, 0, None) == _lib_status("WORKSPACE")
        assert lib.sru_amd_product_grad(dtype, rows, inner, cols, FAKE, FAKE, _lib.F64, FAKE, FAKE, 1 << 40, None) == _lib_status("BAD_DTYPE")


def test_every_product_kernel_in_the_library_can_be_chosen():
    # (rows and columns of the tile in 32, parts of the inner dimension; float splits small tiles only: larger ones start
    # at 384 workgroups, and a split wants at most 256)
    built = set(re.findall(rb"product_tileI(f|NS_9bf16_bitsE|NS_9half_bitsE)Li(\d)ELi(\d)ELi(\d)EEEvNS_13ProductParamsE", open(_lib.LIB_PATH, "rb").read()))
    tiles = {(1, 1, 1), (1, 1, 2), (1, 2, 1), (2, 2, 1)}
    for name, chosen in ((b"f", tiles), (b"NS_9bf16_bitsE", tiles | {(1, 2, 2), (2, 2, 2)}), (b"NS_9half_bitsE", tiles | {(1, 2, 2), (2, 2, 2)})):
        assert {tuple(map(int, b[1:])) for b in built if b[0] == name} == chosen


# Prompts through stacks, us in a graph layer by layer / in chunks of 64 rows / of 32
@pytest.mark.parametrize("length,batch,width,n_proj,layers,taken", [
    (512, 1, 2048, 512, 10, True), (1024, 1, 2048, 512, 10, True),           # 424/286/320, 640/496/628
    (3357, 3, 64, 0, 16, True), (1720, 3, 768, 96, 16, True),                # 1947/495, 1365/1005
    (3550, 3, 2048, 512, 13, False), (3644, 4, 2048, 256, 10, False),        # 2959/6021, 2327/4635
    (998, 4, 2048, 256, 13, False), (1000, 4, 1024, 0, 3, False),            # 997/1659, 208/341
    (996, 3, 768, 0, 3, False), (3996, 4, 1024, 0, 3, False),                # 178/242, 688/1217
    (4096, 4, 2048, 256, 16, False), (4096, 3, 1024, 0, 16, False)])         # workspaces of 1.3 GB and 0.4
def test_prompts_go_by_what_was_measured(length, batch, width, n_proj, layers, taken):
    shape = _lib.Shape(length, batch, width, 1, 3, 0, 1, 0, _lib.BF16, 1, _lib.X_AS_STREAMS)
    nbytes = _lib.load().sru_amd_stack_workspace_bytes(ctypes.byref(shape), layers, n_proj)
    assert (nbytes > 0) == taken and nbytes <= 192 << 20


# One step through stacks, us in a graph layer by layer / in one launch, which is the faster way for all of these launched one by one
@pytest.mark.parametrize("rows,width,n_proj,layers,wanted", [
    (48, 32, 0, 3, 0), (64, 64, 0, 8, 0), (16, 64, 0, 2, 0),          # 21.2/25.3, 51.4/53.5, 18.2/17.6
    (64, 2048, 0, 2, 1), (1, 1024, 0, 2, 1), (16, 256, 0, 8, 1),      # 46.0/44.4, 18.4/18.4
    (48, 64, 32, 3, 1)])
def test_one_step_in_a_graph(rows, width, n_proj, layers, wanted):
    shape = _lib.Shape(1, rows, width, 1, 3, 0, 1, 0, _lib.BF16, 1, _lib.X_AS_STREAMS)
    lib = _lib.load()
    assert lib.sru_amd_stack_workspace_bytes(ctypes.byref(shape), layers, n_proj) > 0
    assert lib.sru_amd_stack_wanted_in_graph(ctypes.byref(shape), layers, n_proj) == wanted
    assert lib.sru_amd_stack_wanted_in_graph(ctypes.byref(shape), 17, n_proj) == 0 and lib.sru_amd_stack_wanted_in_graph(None, layers, n_proj) == 0


def test_a_stacks_call_checks_its_arguments_before_launching():
    lib = _lib.load()
    layers, width, n_proj = 3, 64, 32
    shape = _lib.Shape(1, 4, width, 1, 3, 0, 1, 0, _lib.BF16, 1, _lib.X_AS_STREAMS)
    need = lib.sru_amd_stack_workspace_bytes(ctypes.byref(shape), layers, n_proj)
    pointers = lambda *at: (ctypes.c_void_p * layers)(*(at or [0x1000] * layers))
    # x, weight_proj, weight, weight_c, bias, scale_x, c_init, mask_pad, h, c_last, workspace, its bytes
    fine = dict(x=FAKE, weight_proj=pointers(), weight=pointers(), weight_c=pointers(), bias=pointers(), scale_x=pointers(), c_init=FAKE, mask_pad=FAKE,
                h=FAKE, c_last=FAKE, workspace=FAKE, nbytes=need)

    def call(shape=shape, small16=0, layers=layers, n_proj=n_proj, **kw):
        a = dict(fine, **kw)
        return lib.sru_amd_stack_forward(ctypes.byref(shape) if shape else None, small16, layers, n_proj, *list(a.values())[:-1], a["nbytes"], None)

    code = _lib_status
    assert call(shape=None) == code("NULL_POINTER") and call(workspace=None) == code("WORKSPACE") and call(nbytes=need - 1) == code("WORKSPACE")
    assert call(workspace=ctypes.c_void_p(0x1008)) == code("WORKSPACE")
    for name in ("x", "weight_proj", "weight", "weight_c", "bias", "h", "c_last"):
        assert call(**{name: None}) == code("NULL_POINTER"), name
    for name in ("weight_proj", "weight", "weight_c", "bias"):      # ... and one layer's
        assert call(**{name: pointers(0x1000, None, 0x1000)}) == code("NULL_POINTER"), name
    for name, at in (("x", 0x1008), ("h", 0x1008), ("c_init", 0x1002), ("c_last", 0x1002)):
        assert call(**{name: ctypes.c_void_p(at)}) == code("MISALIGNED"), name
    for name, at in (("weight_proj", 0x1008), ("weight", 0x1008), ("weight_c", 0x1002), ("bias", 0x1002), ("scale_x", 0x1002)):
        assert call(**{name: pointers(0x1000, 0x1000, at)}) == code("MISALIGNED"), name
    every = _lib.SMALL_WEIGHT_C | _lib.SMALL_BIAS | _lib.SMALL_INIT | _lib.SMALL_SCALE | _lib.SMALL_LAST      # 16 bits: two-byte alignment, which leaves x to refuse
    odd = ctypes.c_void_p(0x1002)
    assert call(small16=every, c_init=odd, c_last=odd, weight_c=pointers(*[0x1002] * 3), bias=pointers(*[0x1002] * 3), scale_x=pointers(*[0x1002] * 3),
                x=None) == code("NULL_POINTER")
    assert call(small16=every, weight_c=pointers(0x1001, 0x1000, 0x1000)) == code("MISALIGNED")
    assert call(small16=1 << 20) == code("BAD_FLAGS")
    # what there is no kernel for
    other = lambda **kw: _lib.Shape(*[kw.get(f[0], getattr(shape, f[0])) for f in _lib.Shape._fields_])
    for bad in (other(dtype=_lib.F32), other(k=4, skip_type=2), other(is_custom=1), other(batch=65), other(hidden=48), other(length=2), other(length=64, dirs=2, hidden=32)):
        assert lib.sru_amd_stack_workspace_bytes(ctypes.byref(bad), layers, n_proj) == 0
        assert call(shape=bad) == code("BAD_SHAPE")
    for n, p in ((1, n_proj), (17, n_proj), (-1, n_proj), (layers, -32), (layers, 64), (layers, 33)):
        assert lib.sru_amd_stack_workspace_bytes(ctypes.byref(shape), n, p) == 0 and call(layers=n, n_proj=p) == code("BAD_SHAPE")
    assert call(shape=other(dirs=3)) == code("BAD_FLAGS") and call(shape=other(batch=0)) == code("BAD_SHAPE")
