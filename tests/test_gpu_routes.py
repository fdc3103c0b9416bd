"""One GEMM kernel at a time: a context made under SOKLYN_GEMM_ROUTE runs its GEMMs on the kernel
named there or fails, so what passes has run it, whatever the planner would have chosen.  Against
the oracle, gates as everywhere (tests/helpers.py)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from soklyn_amd import abi
from tests.helpers import FP16_TOL, FP32_TOL, check, rng
from tests.test_gpu_parity import dev, inputs, make_pair

pytestmark = pytest.mark.gpu


@pytest.fixture
def on(ctx, monkeypatch):
    """on(route): a context whose GEMMs take that kernel, on ctx's stream."""
    made = []

    def make(route):
        monkeypatch.setenv("SOKLYN_GEMM_ROUTE", route)
        c = abi.Context(0, 16)
        monkeypatch.delenv("SOKLYN_GEMM_ROUTE")
        c.set_stream(torch.cuda.current_stream().cuda_stream)
        made.append(c)
        return c
    yield make
    torch.cuda.synchronize()
    for c in made:
        c.close()


def dw(ctx, route_ctx, half, M, K, N, saturate=False):
    """The weight gradient and its optimiser step on route_ctx, everything before it on ctx."""
    ob, db = make_pair(ctx, K, N, M, seed=M + K + N, half=half, act=abi.ACT_IDENTITY)
    x = inputs(91, M, K, half)
    xd = dev(x, half)
    s = (rng(92).standard_normal((M, N)) * 512).astype(np.float32)
    if saturate:
        s[:, rng(93).choice(N, size=max(1, N // 8), replace=False)] *= 400.0   # beyond the fp16 range
    ob.forward(x, M)
    ob.error_from_sum(s, M)
    db.forward(xd, M)
    db.error_from_sum(torch.from_numpy(s).cuda(), M)
    if saturate:
        assert torch.isinf(db.d_prenorm_h).any()
    db.ctx = route_ctx
    opt, oopt = (abi.adam(), O.Optimiser.adam()) if half else (abi.sgd(0.5), O.Optimiser.sgd(0.5))
    db.backward(xd, abi.train_ctx(opt, opt, M, 1e-3), 1)
    torch.cuda.synchronize()
    ob.backward(x, oopt, oopt, M, 1e-3, 3.4e38, 1)
    for name in ("dm_w", "dv_w", "dm_b") if half else ("dv_w", "dv_b", "w"):
        check(name, db.get(name), getattr(ob, name), FP16_TOL if half else FP32_TOL)


# the streaming dW: one column and 16, inputs short of, at and past a workgroup's 256, batches
# of one row, part of a 32- or 64-row step, several slices with a short last one
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (3, 255, 16), (33, 256, 7), (65, 257, 10), (200, 31, 3), (4100, 530, 13),
                                   (2049, 1024, 16)])
def test_streaming_dw(ctx, on, half, M, K, N):
    dw(ctx, on("skinny"), half, M, K, N)


def test_streaming_dw_where_d_prenorm_saturates_fp16(ctx, on):
    dw(ctx, on("skinny"), True, 700, 300, 11, saturate=True)


def test_a_kernel_that_does_not_take_the_gemm_is_an_error(ctx, on):
    _, db = make_pair(ctx, 64, 32, 16, seed=1)
    db.ctx = on("skinny")
    with pytest.raises(abi.SklError):
        db.forward(dev(inputs(1, 16, 64, False), False), 16)
