"""One GEMM kernel at a time: a context made under SOKLYN_GEMM_ROUTE runs its GEMMs on the kernel
named there or fails, so what passes has run it, whatever the planner would have chosen.  Against
the oracle, gates as everywhere (tests/helpers.py)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from soklyn_amd import abi
from tests.helpers import FP16_TOL, FP32_TOL, check, f16, rng
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


# ---- the K-splitting kernel -----------------------------------------------------------------
# every tile and count of waves that it is built for: fp16 rows on 4-byte boundaries, fp16 rows at
# odd pitches (through registers), fp32
WAVES = ([(True, 0, f"wave:{r}") for r in ("16:16", "32:4", "64:4", "64:2")] +
         [(True, 1, f"wave:{r}") for r in ("16:16", "32:8", "64:4")] +
         [(False, 0, f"wave:{r}") for r in ("16:16", "32:8", "64:8", "64:4", "64:2", "64:1")])
# short of, at and past the edge of each tile in every dimension; fewer k-tiles than waves, a k-tile
# per wave and stage and more (2114 k: 34 k-tiles of fp16, 67 of fp32), a cut last one; odd: one less
SHAPES = [(2, 2, 2), (16, 64, 32), (17, 66, 34), (64, 128, 64), (65, 130, 66), (130, 2114, 72), (2200, 34, 130)]


@pytest.mark.parametrize("half,odd,route", WAVES)
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_wave_layer(ctx, on, half, odd, route, M, K, N):
    K, N = K - odd, N - odd
    ob, db = make_pair(on(route), K, N, M, seed=M + K, half=half, act=abi.ACT_SILU, p=0.2)
    x = inputs(94, M, K, half)
    tol = FP16_TOL if half else FP32_TOL
    ob.forward(x, M, True, 5)
    db.forward(dev(x, half), M, True, 5)
    torch.cuda.synchronize()
    for name in ("preact", "predrop", "out"):
        check(name, db.get(name), getattr(ob, name), tol)
    assert (db.get("mask") == ob.mask).all()
    s = (rng(95).standard_normal((M, N)) * 512).astype(np.float32)
    ob.error_from_sum(s, M)
    db.error_from_sum(torch.from_numpy(s).cuda(), M)
    check("dx", db.input_grad(M).cpu().numpy(), ob.input_grad(M), tol)


# whole (with the parameter update in the launch; one wave per tile has no room for it) and in slices
# of the batch, the last one short
@pytest.mark.parametrize("half,odd,route", WAVES)
@pytest.mark.parametrize("M,K,N,slices", [(2, 2, 2, 1), (65, 34, 18, 1), (130, 66, 130, 1), (2200, 72, 66, 1),
                                          (2200, 130, 66, 3), (515, 34, 72, 5), (2114, 18, 10, 16)])
def test_wave_dw(ctx, on, half, odd, route, M, K, N, slices):
    if route == "wave:64:1" and slices == 1:
        route = "wave:64:2"
    dw(ctx, on(f"{route}:{slices}"), half, M, K - odd, N - odd)


# an element whose fp16 sum is not finite is summed again in fp32, at its own row and column
# whatever the reduction's or the epilogue's width: rows of 4-element groups, of 2 and odd ones, in
# slices and whole
@pytest.mark.parametrize("route", ["wave:16:16:1", "wave:32:8:1", "wave:64:4:1", "wave:16:16:5", "wave:64:4:7"])
@pytest.mark.parametrize("M,K,N", [(4100, 64, 35), (1500, 33, 65)])
def test_wave_dw_where_d_prenorm_saturates_fp16(ctx, on, route, M, K, N):
    dw(ctx, on(route), True, M, K, N, saturate=True)


@pytest.mark.parametrize("route", ["wave:16:16:1", "wave:32:4:1", "wave:64:2:1", "wave:32:4:5", "wave:64:4:7"])
@pytest.mark.parametrize("M,K,N", [(5000, 130, 10), (1400, 66, 72)])
def test_wave_dw_of_even_rows_where_d_prenorm_saturates_fp16(ctx, on, route, M, K, N):
    dw(ctx, on(route), True, M, K, N, saturate=True)


# the hidden error in its epilogue: the tile's edges, rows past the batch, odd k
@pytest.mark.parametrize("half,odd,route", WAVES)
@pytest.mark.parametrize("M,N0,N1,norm,p", [(2, 4, 2, abi.NORM_RMS, 0.0), (65, 68, 34, abi.NORM_LAYER, 0.1),
                                            (130, 132, 130, abi.NORM_BATCH, 0.0),
                                            (70, 36, 2114, abi.NORM_DISABLED, 0.2)])
def test_wave_hidden_error(ctx, on, half, odd, route, M, N0, N1, norm, p):
    # odd rows have one count of waves per tile; the dW on the same context (its column sums are
    # the error's) has even rows and its own
    N1, K0, c = N1 - odd, 24, on(route.rsplit(":", 1)[0] if odd else route)
    o0, d0 = make_pair(ctx, K0, N0, M, seed=M + N0, half=half, norm=norm, act=abi.ACT_SILU, p=p)
    o1, d1 = make_pair(ctx, N0, N1, M, seed=N1, half=half)
    x = inputs(96, M, K0, half)
    o0.forward(x, M, p > 0, 99)
    d0.forward(dev(x, half), M, p > 0, 99)
    s = (rng(97).standard_normal((M, N1)) * 64).astype(np.float32)
    o1.d_prenorm[:M] = f16(s) if half else s
    d1.d_prenorm.copy_(torch.from_numpy(s))
    if half:
        d1.d_prenorm_h.copy_(torch.from_numpy(s))
    o0.hidden_error(o1, M)
    d0.ctx = c
    d0.hidden_error(d1, M)
    if route == "wave:64:1":
        d0.ctx = ctx     # one wave per tile has no room for the parameter update
    o0.backward(x, O.Optimiser.sgd(0.5), O.Optimiser.sgd(0.5), M, 1e-3, 3.4e38, 1)
    d0.backward(dev(x, half), abi.train_ctx(abi.sgd(0.5), abi.sgd(0.5), M, 1e-3), 1)
    torch.cuda.synchronize()
    names = ["grad", "d_prenorm", "dv_w"] + (["dv_b"] if norm != abi.NORM_BATCH else [])
    names += ["d_norm_w", "d_norm_b", "dv_norm_w"] if norm else []
    names += ["dv_norm_b"] if norm >= abi.NORM_LAYER else []
    for name in names:
        check(name, d0.get(name), getattr(o0, name), FP16_TOL if half else FP32_TOL)


# ---- the register-staged kernels -------------------------------------------------------------
# dW whole and in slices, 16-byte rows and rows read element by element, fp32 tiles of 64 and 128
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,K,N", [(256, 128, 160), (4096, 512, 512), (2500, 300, 130), (1100, 777, 1531),
                                   (130, 65, 33), (100, 1700, 1800)])
def test_staged_dw(ctx, on, half, M, K, N):
    dw(ctx, on("staged"), half, M, K, N)


@pytest.mark.parametrize("M,K,N", [(256, 128, 160), (4096, 512, 512), (2500, 300, 131)])
def test_staged_dw_where_d_prenorm_saturates_fp16(ctx, on, M, K, N):
    dw(ctx, on("staged"), True, M, K, N, saturate=True)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (130, 65, 33), (300, 200, 520), (2100, 129, 1540)])
def test_staged_layer(ctx, on, half, M, K, N):
    test_wave_layer(ctx, on, half, 0, "staged", M, K, N)


# ---- the direct-to-LDS kernel on whole tiles, operands padded where they are not --------------
@pytest.mark.parametrize("M,K,N", [(4096, 3000, 3072), (4096, 3072, 3072)])   # A (and dX's W) padded; none
def test_dma_layer(ctx, on, M, K, N):
    test_wave_layer(ctx, on, True, 0, "dma", M, K, N)


# split-K: whole tiles read in place, padded ones
@pytest.mark.parametrize("M,K,N", [(2048, 2048, 2048), (3000, 1500, 1531)])
def test_dma_dw(ctx, on, M, K, N):
    dw(ctx, on("dma"), True, M, K, N)
