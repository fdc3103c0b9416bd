"""BatchNorm forward (one launch: a workgroup per 16 columns; two launches: column statistics
per row slice, then the outputs) against the oracle at the edges of their row steps and
slices: batches held in registers and not, the last step or slice partly filled, more slices
than fit in registers, widths that are not whole tiles or whole 4-element groups, and bases
off a 16-byte boundary.  The one-launch form over long batches runs under capture, where no
scratch is taken, and gives the two launches' results bit for bit."""
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


OUTS = ("prenorm", "centered", "norm_rstd", "preact", "predrop", "out", "mask")


def eager_and_captured(db, xd, M):
    """The outputs of one forward eagerly and of a graph of it (replayed twice)."""
    db.forward(xd, M, True, 1234)
    torch.cuda.synchronize()
    eager = {n: getattr(db, n).clone() for n in OUTS}
    db.forward(xd, M, True, 7)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        db.forward(xd, M, True, 1234)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
    return eager, {n: getattr(db, n).clone() for n in OUTS}


# the slices of 64 rows (up to 4096) and of 256, a last slice of one row, 16 slices (a pass of the
# one launch's waves) and one more, more than it keeps in LDS, rows with and without 4-element groups
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("M,N,off", [(385, 20, 0), (449, 65, 1), (1024, 16, 0), (1025, 40, 0), (2048, 132, 0),
                                     (4096, 7, 0), (4097, 24, 0), (5000, 33, 2), (65536, 8, 0), (66000, 12, 0),
                                     (70001, 5, 0)])
def test_captured_forward_gives_the_eager_bits(ctx, half, M, N, off):
    _, db = make_pair(ctx, 24, N, M, seed=M + N, half=half, norm=abi.NORM_BATCH, act=abi.ACT_SILU, p=0.25)
    if off:
        misalign(db, off)
    eager, captured = eager_and_captured(db, dev(inputs(72, M, 24, half), half), M)
    for n in OUTS:
        assert torch.equal(eager[n], captured[n]), f"{n} differs between the eager and the captured forward"


# more row blocks than a grid's second dimension holds
def test_a_batch_of_over_four_million_rows(ctx):
    M, N = 4 * 1024 * 1024 + 65, 1
    _, db = make_pair(ctx, 2, N, M, seed=3, norm=abi.NORM_BATCH, act=abi.ACT_IDENTITY)
    g = torch.Generator(device="cuda").manual_seed(5)
    db.forward(torch.randn((M, 2), generator=g, device="cuda"), M)
    torch.cuda.synchronize()
    z = db.prenorm.double()
    mean, var = z.mean(0), z.var(0, unbiased=False)
    assert float((db.centered.double() - (z - mean)).abs().max()) <= FP32_TOL
    assert abs(float(db.norm_rstd[0]) * float((var + 1e-6).sqrt()[0]) - 1.0) <= FP32_TOL
    assert float((db.out.double() - (z - mean) * (var + 1e-6).rsqrt()).abs().max()) <= FP32_TOL


# one context whose stream changes from call to call with nothing waited for: the scratch is one
# for all of them
def test_forwards_of_one_context_on_many_streams(ctx):
    M, N, K = 2048, 256, 32
    here = torch.cuda.current_stream()
    c = abi.Context(0, 16)
    c.set_sync(False)
    pairs = [make_pair(c, K, N, M, seed=i, half=True, norm=abi.NORM_BATCH, act=abi.ACT_SILU)[1] for i in range(12)]
    xs = [dev(inputs(i, M, K, True), True) for i in range(12)]
    c.set_stream(here.cuda_stream)
    want = []
    for db, x in zip(pairs, xs):
        db.forward(x, M)
        torch.cuda.synchronize()
        want.append(db.out.clone())
        db.out.zero_()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    for rep in range(3):
        for i, (db, x) in enumerate(zip(pairs, xs)):
            c.set_stream(streams[(i + rep) % 4].cuda_stream)
            db.forward(x, M)
    torch.cuda.synchronize()
    for db, w in zip(pairs, want):
        assert torch.equal(db.out, w)
    c.set_stream(here.cuda_stream)
    c.close()


# a context's first long-batch forward while another stream is captured in the global mode, which
# an allocation of this thread's would end
def test_first_forward_beside_a_capture(ctx):
    M, N, K = 1024, 64, 32
    here, other = torch.cuda.current_stream(), torch.cuda.Stream()
    _, db = make_pair(ctx, K, N, M, seed=8, half=True, norm=abi.NORM_BATCH, act=abi.ACT_SILU)
    x = dev(inputs(9, M, K, True), True)
    db.forward(x, M)
    torch.cuda.synchronize()
    want = db.out.clone()
    c = abi.Context(0, 16)
    c.set_stream(other.cuda_stream)
    c.set_sync(False)
    a, graph = torch.zeros(64, device="cuda"), torch.cuda.CUDAGraph()
    db.ctx = c
    with torch.cuda.graph(graph, stream=here):
        a.add_(1.0)
        db.forward(x, M)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(db.out, want) and bool((a == 1.0).all())
    db.ctx = ctx
    c.close()
