"""Softmax and cross-entropy error of the output layer (one launch up to 64 classes without a
norm, two beyond) against the oracle at the edges of its lanes per row and rows per step, with
rows of the cache past the targets (softmax alone), and the column sums it leaves for the
bias update."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from soklyn_amd import abi
from tests.helpers import FP16_TOL, FP32_TOL, rng
from tests.test_gpu_parity import check, dev, inputs, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N", [(1, 1), (3, 2), (100, 10), (33, 16), (33, 17), (65, 32), (65, 33), (70, 64), (9, 65),
                                 (300, 1000), (20000, 3)])
def test_softmax_ce(ctx, half, M, N):
    K, extra = 8, 5
    ob, db = make_pair(ctx, K, N, M + extra, seed=M + N, half=half)
    x = inputs(91, M, K, half)
    ob.forward(x, M)
    db.forward(dev(x, half), M)
    t = np.zeros((M, N), np.float32)
    t[np.arange(M), rng(92).integers(0, N, M)] = 1.0
    print(f"softmax + CE {M}x{N} half={half}", flush=True)
    ob.output_error(t, abi.LOSS_CE, abi.ACT_SOFTMAX)
    db.output_error(dev(t, half), abi.LOSS_CE, abi.ACT_SOFTMAX)
    tol = FP16_TOL if half else FP32_TOL
    check("out", db.get("out"), ob.out, tol)
    if N > 1:   # one class: every error is 0
        for name in ("grad", "d_prenorm"):
            check(name, db.get(name)[:M], getattr(ob, name)[:M], tol)
    if half:
        assert np.array_equal(db.get("d_prenorm_h"), db.get("d_prenorm").astype(np.float16).astype(np.float32))
    # the bias gradient from the column sums: close to the sum of the device's own errors
    opt = abi.sgd(0.0)
    db.backward(dev(x, half), abi.train_ctx(opt, opt, M, 1e-3), 1)
    torch.cuda.synchronize()
    dp = db.get("d_prenorm")[:M].astype(np.float64)
    bound = np.abs(dp).sum(0) * M * 2.0 ** -24 + 1e-30   # n u sum|terms|, any order of n additions
    got = db.get("dv_b").reshape(-1).astype(np.float64) * 512 * M
    # (two more roundings: the scale and the mean)
    assert np.all(np.abs(got - dp.sum(0)) <= bound + 2.0 ** -22 * np.abs(dp.sum(0)))
