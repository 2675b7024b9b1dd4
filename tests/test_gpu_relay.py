"""The forward kernel for few columns (sru_relay.h) against the CPU oracle: walks around its chunk of 16
steps and past the lengths from which it is taken (64 and 128 steps, 40 more with a mask), column counts
that do not fill its last workgroup of 64, workgroups across directions and batch rows, the column limit.
Tolerances and the backward pass from its checkpoints as in test_gpu_parity.py."""
import numpy as np
import pytest
import torch

import sru_amd
from tests.abi import DeviceProblem
from tests.cases import Case
from tests.test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    dict(L=168, B=1, d=8),
    dict(L=169, B=3, d=24, dirs=2, pad="right", scale=1.7),
    dict(L=175, B=5, d=152, dirs=2, pad="right", mask_c=True),
    dict(L=176, B=2, d=64, dirs=2, k=4, pad="random"),
    dict(L=177, B=9, d=16, dirs=2, k=4, act=1),
    dict(L=183, B=2, d=128, skip=False, pad="right", mask_c=True),
    dict(L=191, B=3, d=40, dirs=2, act=1, pad="random", scale=1.3),
    dict(L=192, B=4, d=2048, dirs=2, zero_c0=True),
]


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cfg", SHAPES, ids=lambda g: "-".join(f"{k}{v}" for k, v in g.items()))
def test_against_the_oracle(cfg, dt):
    check_against_oracle(Case(seed=31, **cfg), dt, checkpointed=True)
    check_against_oracle(Case(seed=32, **cfg), dt, keep_c=False)


@pytest.mark.parametrize("pad", [None, "right"])
def test_float_x_beside_16_bit_streams(pad):
    check_against_oracle(Case(L=169, B=3, d=72, dirs=2, scale=1.7, mask_c=True, pad=pad, seed=33), "bf16",
                         checkpointed=True, x_f32=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_padding_is_not_touched_by_what_it_holds(dtype):
    # NaN and infinities in padded cells, an infinite state carried over padding, a row that is all padding
    L, B, d = 180, 4, 32
    gen = torch.Generator().manual_seed(1)
    u = torch.randn(L, B, 6 * d, generator=gen).to(dtype)
    x = torch.randn(L, B, 2 * d, generator=gen).to(dtype)
    pad = torch.zeros(L, B, dtype=torch.bool)
    pad[100:, 1] = True
    pad[:, 2] = True
    pad[50:70, 3] = True
    c0 = torch.randn(B, 2 * d, generator=gen)
    c0[2, 5], c0[2, 6], c0[2, 7] = float("inf"), float("-inf"), float("nan")
    clean_u, clean_x = u.clone(), x.clone()
    u[pad], x[pad] = float("nan"), float("inf")
    wc, bias = torch.randn(4 * d, generator=gen), torch.randn(4 * d, generator=gen)
    run = lambda a, b: [t.cpu() for t in sru_amd.elementwise_recurrence_inference(
        a.cuda(), b.cuda(), wc.cuda(), bias.cuda(), c0.cuda(), 0, d, True, True, None, None, pad.cuda())]
    (h, last), (h0, last0) = run(u, x), run(clean_u, clean_x)
    assert torch.equal(h, h0) and not h.isnan().any()
    assert torch.equal(last.nan_to_num(nan=7.0), last0.nan_to_num(nan=7.0))
    assert (h[pad] == 0).all()
    assert np.array_equal(last[2].float().numpy(), c0[2].to(last.dtype).float().numpy(), equal_nan=True)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("B", [256, 257])
def test_column_limit(B, dt):
    # the last 64 columns that it takes, and a batch row more, which the other kernels take
    from torch.profiler import ProfilerActivity, profile
    case = Case(L=130, B=B, d=64, seed=34)
    check_against_oracle(case, dt, keep_c=False)
    dp = DeviceProblem(case, dt, checkpointed=True)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        dp.forward()
        torch.cuda.synchronize()
    scans = [e.name for e in seen.events() if "forward_scan" in e.name]
    assert len(scans) == 1 and ("forward_scan_relay" in scans[0]) == (B == 256)
