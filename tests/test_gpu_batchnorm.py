"""BatchNorm forward (one launch: a workgroup per 16 columns; two launches: column statistics
per row slice, then the outputs) against the oracle at the edges of their row steps and
slices: batches held in registers and not, the last step or slice partly filled, more slices
than fit in registers, widths that are not whole tiles or whole 4-element groups, and bases
off a 16-byte boundary.  The one-launch form over long batches runs under capture, where no
scratch is taken."""
from __future__ import annotations

import pytest
import torch

from soklyn_amd import abi
from tests.helpers import FP16_TOL, FP32_TOL
from tests.test_gpu_parity import check, dev, inputs, make_pair
from tests.test_gpu_unaligned import misalign

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,off", [
    (2, 16, 0), (64, 40, 0), (257, 20, 0), (512, 132, 0), (513, 48, 0), (2048, 16, 0), (2049, 24, 0), (5000, 12, 0),
    (70, 13, 0), (513, 33, 0), (2049, 7, 0), (300, 32, 1), (300, 32, 2), (385, 68, 0), (449, 65, 1), (4097, 72, 0),
    (16700, 20, 0), (4100, 3, 0)])
@pytest.mark.parametrize("captured", [False, True])
def test_batchnorm_forward(ctx, half, M, N, off, captured):
    if captured and M <= 384:
        pytest.skip("short batches take the same launch either way")
    K = 32
    ob, db = make_pair(ctx, K, N, M, seed=M + N, half=half, norm=abi.NORM_BATCH, act=abi.ACT_SILU, p=0.25)
    if off:
        misalign(db, off)
    x = inputs(71, M, K, half)
    ob.forward(x, M, True, 1234)
    xd = dev(x, half)
    if captured:
        db.forward(xd, M, True, 7)   # other values in every output, and nothing left to load
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
            db.forward(xd, M, True, 1234)
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
    else:
        db.forward(xd, M, True, 1234)
    torch.cuda.synchronize()
    # two rows: the variance is (z1 - z0)^2 / 4, so a relative error of a small difference
    # of the fp16-rounded prenorm goes into every result of its column
    tol = FP16_TOL if half else FP32_TOL
    for name in ("prenorm", "centered", "norm_rstd", "preact", "predrop", "out"):
        if M == 2 and name != "prenorm" and half:
            continue
        check(f"{name} {M}x{N}", db.get(name).reshape(-1)[:N] if name == "norm_rstd" else db.get(name),
              getattr(ob, name).reshape(-1)[:N] if name == "norm_rstd" else getattr(ob, name), tol)
    assert (db.get("mask") == ob.mask).all()
