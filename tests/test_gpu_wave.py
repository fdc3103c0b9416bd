"""A layer's step at sizes whose GEMMs the planner gives mostly to the K-splitting kernel (16x16,
32x32 and 64x64 tiles, each wave its own k-tiles), against the oracle: sizes around the edges
of its tiles and k-tiles, fewer k-tiles than waves, widths that are odd (fp16 rows through
registers), even but not whole 16-byte chunks (the last chunk of a row masked); outputs and
inputs off a 16-byte boundary.  Which tile, or which other kernel, a size takes is the
planner's choice; tests/test_gpu_routes.py runs each by name.  Gates as everywhere
(tests/helpers.py)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from soklyn_amd import abi
from tests.helpers import FP16_TOL, FP32_TOL, check_adam_update, f16, rng
from tests.test_gpu_fused_error import test_fused_hidden_error_and_backward as fused_error
from tests.test_gpu_parity import check, dev, inputs, make_pair
from tests.test_gpu_unaligned import misalign

pytestmark = pytest.mark.gpu

SHAPES = [  # batch, inputs, outputs
    (1, 1, 1), (2, 3, 5), (16, 64, 16), (17, 65, 33), (15, 63, 31), (64, 128, 64), (33, 130, 66), (5, 1000, 24),
    (70, 77, 200), (130, 36, 12), (20, 4100, 10), (257, 520, 136),
    (700, 72, 900), (515, 330, 902), (701, 129, 835),      # several hundred tiles
    (1700, 40, 2000), (2500, 33, 2560), (2000, 1700, 40),  # more than one round of them
    (3001, 200, 96), (4100, 61, 35), (5000, 130, 10), (2053, 40, 3),   # long batches under few tiles of dW
]


def step(ctx, half, M, K, N, off=0, x_off=0):
    ob, db = make_pair(ctx, K, N, M, seed=M + K + N, half=half, act=abi.ACT_SILU)
    if off:
        misalign(db, off)
    w0 = (db.get("master_w") if half else db.get("w")).copy()
    x = inputs(81, M, K, half)
    xd = dev(x, half)
    if x_off:
        buf = torch.zeros(xd.numel() + 8, device="cuda", dtype=xd.dtype)
        view = buf[x_off:x_off + xd.numel()].view(xd.shape)
        view.copy_(xd)
        xd = view
    s = (rng(82).standard_normal((M, N)) * 512).astype(np.float32)
    print(f"step {M}x{K}->{N} half={half} off={off},{x_off}", flush=True)
    ob.forward(x, M)
    db.forward(xd, M)
    ob.error_from_sum(s, M)
    db.error_from_sum(torch.from_numpy(s).cuda(), M)
    dx = db.input_grad(M).cpu().numpy()
    opt = abi.sgd(0.5) if not half else abi.adam()
    db.backward(xd, abi.train_ctx(opt, opt, M, 1e-3), 1)
    torch.cuda.synchronize()
    ref_dx = ob.input_grad(M)
    oopt = O.Optimiser.adam() if half else O.Optimiser.sgd(0.5)
    ob.backward(x, oopt, oopt, M, 1e-3, 3.4e38, 1)
    tol = FP16_TOL if half else FP32_TOL
    for name in ("preact", "predrop", "out"):
        check(name, db.get(name), getattr(ob, name), tol)
    check("dx", dx, ref_dx, tol)
    m = "dm" if half else "dv"
    for name in (f"{m}_w", f"{m}_b"):
        check(name, db.get(name), getattr(ob, name), tol)
    if half:
        # Adam's first step is lr sign(g) whatever |g| is: where g is rounding noise the
        # sign is, too, so the update is checked against the device's own moments
        check_adam_update("w", w0, db.get("master_w"), db.get("dm_w"), db.get("dv_w"), 1e-3, 1,
                          np.asarray(ob.master_w).reshape(K, N) - w0, np.asarray(ob.dm_w).reshape(K, N))
        assert (db.get("w") == f16(db.get("master_w"))).all()
    else:
        check("w", db.get("w"), ob.w, tol)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_step(ctx, half, M, K, N):
    step(ctx, half, M, K, N)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("off,x_off", [(1, 0), (2, 1), (0, 1), (0, 2), (0, 3)])
def test_step_misaligned(ctx, half, off, x_off):
    step(ctx, half, 50, 96, 72, off, x_off)


# fp16 grids on 128x128 direct-to-LDS tiles short of the 256x256 kernel's: the forward, the
# input gradient and, in the hidden error, the fused epilogue


def test_step_128(ctx):
    step(ctx, True, 2048, 1024, 2048)


# ... and on operands as stored: ragged M and N, an odd number of k-tiles whose last is cut,
# rows of the output that are whole vectors, 4-element groups, and neither
@pytest.mark.parametrize("M,K,N", [(2100, 2104, 2056), (2049, 2184, 2052), (2177, 2120, 2050)])
def test_step_ragged_128(ctx, M, K, N):
    step(ctx, True, M, K, N)


@pytest.mark.parametrize("norm,act,p", [(abi.NORM_RMS, abi.ACT_MISH, 0.1), (abi.NORM_BATCH, abi.ACT_TANH, 0.0)])
def test_hidden_error_128(ctx, norm, act, p):
    fused_error(ctx, 2048, 64, 2048, 1024, norm, act, p, 0)


# the hidden error in the K-splitting kernel's epilogue: each tile, rows past the batch, columns
# past the output, odd k (fp16 rows through registers), every norm; its column sums through the
# bias and norm-parameter moments.  A width that is not whole 4-column groups takes two kernels.
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N0,N1,norm,act,p", [
    (3, 4, 17, abi.NORM_RMS, abi.ACT_MISH, 0.0), (40, 36, 33, abi.NORM_LAYER, abi.ACT_SILU, 0.1),
    (130, 100, 200, abi.NORM_BATCH, abi.ACT_TANH, 0.0), (257, 516, 66, abi.NORM_DISABLED, abi.ACT_SILU, 0.2),
    (515, 900, 330, abi.NORM_RMS, abi.ACT_MISH, 0.1), (701, 836, 129, abi.NORM_LAYER, abi.ACT_SIGMOID, 0.0),
    (1700, 2000, 40, abi.NORM_DISABLED, abi.ACT_TANH, 0.0), (66, 50, 72, abi.NORM_RMS, abi.ACT_SILU, 0.0)])
def test_hidden_error(ctx, half, M, N0, N1, norm, act, p):
    K0 = 24
    print(f"hidden error M={M} {N0} <- {N1} norm={norm} half={half}", flush=True)
    o0, d0 = make_pair(ctx, K0, N0, M, seed=M + N0, half=half, norm=norm, act=act, p=p)
    o1, d1 = make_pair(ctx, N0, N1, M, seed=N1, half=half)
    x = inputs(111, M, K0, half)
    o0.forward(x, M, p > 0, 99)
    d0.forward(dev(x, half), M, p > 0, 99)
    o1.forward(o0.out, M)
    d1.forward(d0.out, M)
    s = (rng(112).standard_normal((M, N1)) * 64).astype(np.float32)
    o1.error_from_sum(s, M)
    d1.error_from_sum(torch.from_numpy(s).cuda(), M)
    opt = (O.Optimiser.sgd(0.5), abi.sgd(0.5))
    o0.hidden_error(o1, M)
    o0.backward(x, opt[0], opt[0], M, 1e-3, 3.4e38, 1)
    d0.backward_hidden(d1, dev(x, half), abi.train_ctx(opt[1], opt[1], M, 1e-3), 1)
    torch.cuda.synchronize()
    tol = FP16_TOL if half else FP32_TOL
    for name in ["grad", "d_prenorm"] + (["d_norm_w", "d_norm_b"] if norm else []):
        check(name, d0.get(name), getattr(o0, name), tol)
    if half:
        assert np.array_equal(d0.get("d_prenorm_h"), f16(d0.get("d_prenorm")))
    names = (["dv_b"] if norm != abi.NORM_BATCH else []) + (["dv_norm_w"] if norm else [])
    names += ["dv_norm_b"] if norm >= abi.NORM_LAYER else []
    for name in names + ["dv_w"]:
        check(name, d0.get(name), getattr(o0, name), tol)


# the layer above of at most 16 outputs: in the epilogue of small layers, in the error kernel
# of larger ones and for widths that are not whole 4-column groups
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N0,N1,norm", [(1, 4, 1, abi.NORM_DISABLED), (64, 128, 10, abi.NORM_DISABLED),
                                          (300, 260, 3, abi.NORM_RMS), (1024, 512, 16, abi.NORM_LAYER),
                                          (2048, 1024, 10, abi.NORM_RMS), (2049, 1024, 10, abi.NORM_RMS),
                                          (130, 51, 7, abi.NORM_BATCH)])
def test_hidden_error_below_a_narrow_layer(ctx, half, M, N0, N1, norm):
    test_hidden_error(ctx, half, M, N0, N1, norm, abi.ACT_SILU, 0.1)


# Layers whose backward buffers are one piece of memory, and a narrow layer fed its own output:
# the calls that read and write it take routes that read it whole first.
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N0,N1", [(512, 512, 256), (300, 260, 72)])
def test_hidden_error_over_the_layer_above(ctx, half, M, N0, N1):
    K0 = 24
    o0, d0 = make_pair(ctx, K0, N0, M, seed=M + N0, half=half, act=abi.ACT_SILU)
    o1, d1 = make_pair(ctx, N0, N1, M, seed=N1, half=half)
    # one buffer of the larger size: d0's whole, d1's a leading part of it
    name = "d_prenorm_h" if half else "d_prenorm"
    setattr(d1, name, getattr(d0, name).view(-1)[:M * N1].view(M, N1))
    x = inputs(111, M, K0, half)
    o0.forward(x, M)
    d0.forward(dev(x, half), M)
    o1.forward(o0.out, M)
    d1.forward(d0.out, M)
    s = (rng(112).standard_normal((M, N1)) * 64).astype(np.float32)
    o1.error_from_sum(s, M)
    d1.error_from_sum(torch.from_numpy(s).cuda(), M)
    o0.hidden_error(o1, M)
    d0.hidden_error(d1, M)
    torch.cuda.synchronize()
    for field in ("grad", "d_prenorm"):
        check(field, d0.get(field), getattr(o0, field), FP16_TOL if half else FP32_TOL)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N", [(200, 64), (77, 10)])
def test_forward_of_its_own_output(ctx, half, M, N):
    ob, db = make_pair(ctx, N, N, M, seed=N, half=half, act=abi.ACT_SILU)
    x = inputs(113, M, N, half)
    db.out.copy_(dev(x, half))
    ob.forward(x, M)
    db.forward(db.out, M)
    torch.cuda.synchronize()
    check("out", db.get("out"), ob.out, FP16_TOL if half else FP32_TOL)


# ... and of any width and number of rounds of tiles: a copy of the operand is read
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N", [(300, 520), (2100, 1030), (4096, 1024)])
def test_forward_of_its_own_wide_output(ctx, half, M, N):
    _, db = make_pair(ctx, N, N, M, seed=N, half=half, act=abi.ACT_SILU)
    x = dev(inputs(114, M, N, half), half)
    db.forward(x, M)
    torch.cuda.synchronize()
    want = db.out.clone()
    db.out.copy_(x)
    db.forward(db.out, M)
    torch.cuda.synchronize()
    check("out", db.get("out"), want.float().cpu().numpy(), FP16_TOL if half else FP32_TOL)


# the input gradient over the fp32 operand it is computed from, and over half of it; over the fp16
# copy that an fp16 block's reads
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,K,N", [(320, 200, 200), (300, 520, 520), (1000, 777, 1560), (4096, 1024, 1024)])
def test_input_grad_over_its_operand(ctx, half, M, K, N):
    _, db = make_pair(ctx, K, N, M, seed=K + N, half=half, act=abi.ACT_IDENTITY)
    d = torch.from_numpy((rng(115).standard_normal((M, N)) * 512).astype(np.float32)).cuda()
    db.d_prenorm.copy_(d)
    name = "d_prenorm"
    if half:
        name = "d_prenorm_h"   # room for the fp32 output behind its rows
        db.d_prenorm_h = torch.empty(2 * M * max(K, N), device="cuda", dtype=torch.float16)[:M * N].view(M, N)
        db.d_prenorm_h.copy_(d)
    want = db.input_grad(M).cpu().numpy()
    out = torch.as_strided(getattr(db, name).view(torch.float32) if half else db.d_prenorm, (M, K), (K, 1))
    got = db.input_grad(M, out=out).cpu().numpy()
    check("dx", got, want, FP32_TOL)
