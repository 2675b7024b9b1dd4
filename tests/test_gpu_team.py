"""The backward kernel whose wavefronts share a walk (sru_team.h) against the CPU oracle: walks from its shortest
(17 steps) on, around chunks of 8 steps and rounds of 4 and 8 chunks; columns by direction and row (d near a
multiple of 64), any 64 columns (other d), a last workgroup that is not full; the limits of its column counts.
Tolerances as in test_gpu_parity.py: its sums are those of the other kernels but for the order of a chunk's factors."""
import numpy as np
import pytest
import torch

import sru_amd
from tests.cases import Case
from tests.test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(L=17, B=1, d=8),
    dict(L=24, B=3, d=56, dirs=2, pad="right", scale=1.7),
    dict(L=31, B=5, d=152, dirs=2, pad="right", mask_c=True),
    dict(L=33, B=130, d=64, k=4, pad="random"),
    dict(L=64, B=3, d=120, dirs=2, k=4, act=1),
    dict(L=65, B=2, d=64, dirs=2, skip=False, pad="right", mask_c=True),
    dict(L=72, B=7, d=22, dirs=2, act=1, pad="random", scale=1.3),
    dict(L=128, B=4, d=128, dirs=2, zero_c0=True),
    dict(L=129, B=1, d=40, dirs=2, skip=False, act=1),
    dict(L=201, B=3, d=304, dirs=2, k=4, pad="right"),
]


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cfg", SHAPES, ids=lambda g: "-".join(f"{k}{v}" for k, v in g.items()))
def test_against_the_oracle(cfg, dt):
    check_against_oracle(Case(seed=41, **cfg), dt, checkpointed=True)


@pytest.mark.parametrize("pad", [None, "right"])
@pytest.mark.parametrize("d", [72, 192])
def test_float_x_beside_16_bit_streams(d, pad):
    check_against_oracle(Case(L=57, B=3, d=d, dirs=2, scale=1.7, mask_c=True, pad=pad, seed=42), "bf16",
                         checkpointed=True, x_f32=True)


@pytest.mark.parametrize("dt,B", [("f32", 256), ("f32", 257), ("bf16", 128), ("bf16", 129), ("bf16", 768), ("bf16", 769)])
def test_column_limits(dt, B):
    check_against_oracle(Case(L=41, B=B, d=64, seed=43), dt, checkpointed=True)


@pytest.mark.parametrize("d", [24, 64])
@pytest.mark.parametrize("L", [32, 100])
def test_factors_beyond_the_float_range(L, d):
    # Every step but the first multiplies the state's gradient by about 4e5, eight of them by more than a float
    # holds; the gradient itself is zero there (only the first output has one), and stays zero.
    gen = np.random.default_rng(5)
    B, D = 2, d
    u = np.zeros((L, B, D, 3), np.float32)
    c = np.zeros((B, D), np.float32)
    for t in range(L):
        u[t, ..., 0] = 4e6 * (-1) ** t * (1 + 0.1 * gen.random((B, D)))
        u[t, ..., 1] = 2.0 - c
        g = 1 / (1 + np.exp(-(u[t, ..., 1].astype(np.float64) + c)))
        c = ((c - u[t, ..., 0]) * g + u[t, ..., 0]).astype(np.float32)
    leaf = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda", requires_grad=True)
    U, x = leaf(u.reshape(L, B, 3 * D)), leaf(gen.standard_normal((L, B, D)))
    wc, bias = leaf(np.ones(2 * D)), leaf(np.zeros(2 * D))
    h, _ = sru_amd.ElementwiseRecurrence.apply(U, x, wc, bias, None, 0, d, False, True, None, None, None)
    gh = torch.zeros_like(h)
    gh[0] = 1.0
    gu, gx, gwc, gbias = torch.autograd.grad(h, (U, x, wc, bias), gh)
    gu = gu.view(L, B, D, 3).cpu()
    assert (gu[1:] == 0).all() and (gx[1:] == 0).all()
    # the first step: c = u0 (1 - g1), h = (c - x) g2 + x with g2 = 1/2
    u0, x0 = torch.tensor(u[0, ..., 0]).double(), x[0].detach().cpu().double()
    g1 = torch.sigmoid(torch.tensor(2.0, dtype=torch.float64))
    expect = torch.stack([0.5 * (1 - g1).expand_as(u0), -0.5 * u0 * g1 * (1 - g1), 0.25 * (u0 * (1 - g1) - x0)], -1)
    # (a gate is within 1e-7, relative to 1 - g1 = 0.12: 1e-6)
    assert ((gu[0].double() - expect).abs() <= 2e-6 * expect.abs()).all()
    assert (gwc == 0).all() and gbias.isfinite().all()


# (streams, steps, rows, d, options, taken): both sides of each line of the rule, beyond which other kernels are the faster ones
LINES = [
    ("bf16", 16, 4, 512, {}, False), ("bf16", 17, 4, 512, {}, True), ("bf16", 24, 64, 512, {}, True), ("bf16", 24, 65, 512, {}, False),
    ("f16", 89, 80, 512, {}, True), ("f16", 89, 81, 512, {}, False), ("bf16", 88, 80, 512, {}, False), ("bf16", 89, 80, 512, dict(x_f32=True), False),
    ("bf16", 19, 52, 304, {}, False), ("bf16", 20, 52, 304, {}, True), ("bf16", 127, 102, 304, {}, True), ("bf16", 127, 103, 304, {}, False),
    ("bf16", 128, 76, 304, {}, True), ("bf16", 128, 77, 304, {}, False), ("bf16", 128, 102, 304, dict(pad=True), True), ("bf16", 128, 103, 304, dict(pad=True), False),
    ("bf16", 64, 85, 160, {}, True), ("bf16", 64, 86, 160, {}, False), ("bf16", 63, 170, 160, {}, True), ("bf16", 40, 57, 304, dict(x_f32=True), True),
    ("bf16", 40, 58, 304, dict(x_f32=True), False), ("bf16", 40, 170, 160, dict(x_f32=True), True), ("bf16", 40, 171, 160, dict(x_f32=True), False),
    ("f32", 17, 32, 512, {}, True), ("f32", 17, 33, 512, {}, False), ("f32", 17, 4, 250, {}, False), ("f32", 18, 64, 250, {}, True),
    ("f32", 256, 56, 250, {}, True), ("f32", 256, 57, 250, {}, False), ("f32", 256, 64, 250, dict(pad=True), True), ("f32", 256, 65, 250, dict(pad=True), False),
]


@pytest.mark.parametrize("dt,L,B,d,kw,taken", LINES, ids=lambda v: "-".join(v) if isinstance(v, dict) else str(v))
def test_where_it_is_taken(dt, L, B, d, kw, taken):
    from torch.profiler import ProfilerActivity, profile
    t = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dt]
    leaf = lambda *size, dtype=t: torch.randn(*size, device="cuda", dtype=dtype).requires_grad_()
    u, x = leaf(L, B, 3 * d), leaf(L, B, d, dtype=torch.float32 if "x_f32" in kw else t)
    wc, bias = leaf(2 * d, dtype=torch.float32), leaf(2 * d, dtype=torch.float32)
    pad = torch.zeros(L, B, dtype=torch.bool, device="cuda") if "pad" in kw else None
    h, _ = sru_amd.ElementwiseRecurrence.apply(u, x, wc, bias, None, 0, d, False, True, None, None, pad)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        torch.autograd.grad(h, (u, x, wc, bias), torch.ones_like(h))
        torch.cuda.synchronize()
    scans = [e.name for e in seen.events() if "backward_scan" in e.name]
    assert len(scans) == 1 and ("backward_scan_team" in scans[0]) == taken, scans


# walks of several chunks past those lines: lane pairs on registers and on row tiles, one column per lane
PAST = [("bf16", dict(L=25, B=641, d=64, pad="right", scale=1.7), {}), ("f16", dict(L=41, B=641, d=64, k=4, act=1), {}),
        ("bf16", dict(L=33, B=641, d=64, skip=False, pad="random"), {}), ("bf16", dict(L=27, B=330, d=70, dirs=2, mask_c=True), {}),
        ("bf16", dict(L=25, B=641, d=64, pad="right", scale=1.3), dict(x_f32=True)), ("f16", dict(L=40, B=290, d=70), dict(x_f32=True)),
        ("bf16", dict(L=67, B=110, d=160), {}), ("f16", dict(L=72, B=110, d=160, k=4, act=1, mask_c=True), {}),
        ("bf16", dict(L=64, B=220, d=80, dirs=2, skip=False, pad="random"), {}), ("f32", dict(L=41, B=257, d=64, k=4, act=1, pad="right"), {}),
        ("f32", dict(L=25, B=130, d=64, dirs=2, skip=False, mask_c=True), {})]


@pytest.mark.parametrize("dt,cfg,kw", PAST, ids=lambda v: "-".join(f"{k}{x}" for k, x in v.items()) if isinstance(v, dict) else v)
def test_the_kernels_past_the_lines(dt, cfg, kw):
    check_against_oracle(Case(seed=44, **cfg), dt, checkpointed=True, **kw)


@pytest.mark.parametrize("L,B,d", [(32, 2, 24), (100, 2, 24), (100, 2, 64), (100, 130, 64)])   # teams of 4, 8, 8, 4; up to 4 rounds
def test_gradients_beside_factors_beyond_the_float_range(L, B, d):
    # Every fifth column as in the test above; it has the whole wavefront hand its gradients on step by step. The other
    # columns have ordinary factors, a gradient of every output and of the last state, and 64-bit results.
    gen = np.random.default_rng(6)
    hot = np.arange(d) % 5 == 2
    u = gen.standard_normal((L, B, d, 3)).astype(np.float32)
    wc, bias = gen.uniform(-1.2, 1.2, (2, d)).astype(np.float32), (0.5 * gen.standard_normal((2, d))).astype(np.float32)
    wc[:, hot], bias[:, hot] = 1.0, 0.0
    c = np.zeros((B, d), np.float32)
    for t in range(L):
        h0 = 4e6 * (-1) ** t * (1 + 0.1 * gen.random((B, d)))
        u[t][:, hot, 0], u[t][:, hot, 1] = h0[:, hot], 2.0 - c[:, hot]
        g = 1 / (1 + np.exp(-(u[t, ..., 1].astype(np.float64) + wc[0] * c + bias[0])))
        c = ((c - u[t, ..., 0]) * g + u[t, ..., 0]).astype(np.float32)
    gh, gl = gen.standard_normal((L, B, d)).astype(np.float32), gen.standard_normal((B, d)).astype(np.float32)
    gh[1:, :, hot], gl[:, hot] = 0.0, 0.0
    x = gen.standard_normal((L, B, d)).astype(np.float32)
    leaf = lambda a, kind: torch.tensor(a).to(kind).requires_grad_()
    U, X, W, b = (leaf(a, torch.float32).detach().cuda().requires_grad_() for a in (u.reshape(L, B, 3 * d), x, wc.reshape(-1), bias.reshape(-1)))
    outs = sru_amd.ElementwiseRecurrence.apply(U, X, W, b, None, 0, d, False, True, None, None, None)
    got = [t.cpu().double() for t in torch.autograd.grad(outs, (U, X, W, b), (torch.tensor(gh).cuda(), torch.tensor(gl).cuda()))]
    got = got[0].view(L, B, d, 3), got[1], got[2].view(2, d), got[3].view(2, d)
    assert (got[0][1:, :, hot] == 0).all() and (got[1][1:, :, hot] == 0).all() and all(t.isfinite().all() for t in got)

    cold = torch.tensor(~hot)
    U, X, W, b = leaf(u[:, :, ~hot], torch.float64), leaf(x[:, :, ~hot], torch.float64), leaf(wc[:, ~hot], torch.float64), leaf(bias[:, ~hot], torch.float64)
    state, h = torch.zeros(B, int(cold.sum()), dtype=torch.float64), []
    for t in range(L):
        g1, g2 = torch.sigmoid(U[t, ..., 1] + W[0] * state + b[0]), torch.sigmoid(U[t, ..., 2] + W[1] * state + b[1])
        state = (state - U[t, ..., 0]) * g1 + U[t, ..., 0]
        h.append((state - X[t]) * g2 + X[t])
    want = torch.autograd.grad((torch.stack(h), state), (U, X, W, b), (torch.tensor(gh[:, :, ~hot]).double(), torch.tensor(gl[:, ~hot]).double()))
    for a, r in zip((got[0][:, :, cold], got[1][:, :, cold]), want[:2]):
        assert ((a - r).abs() <= 1e-5 * r.abs().clamp(min=1.0)).all()
    for a, r in zip((got[2][:, cold], got[3][:, cold]), want[2:]):
        assert ((a - r).abs() <= 1e-5 * max(1.0, float(r.abs().max()))).all()
