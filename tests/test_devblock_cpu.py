"""DeviceBlock's per-call descriptors on the CPU: each holds the block's scalars and the
current address of every tensor its call reads, and nothing else; a tensor or a mode changed
between calls is seen."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from soklyn_amd import abi, devblock
from soklyn_amd.devblock import DeviceBlock


class NoContext:
    h = None


def block(half, norm):
    return DeviceBlock(NoContext(), 24, 16, 8, np.zeros((24, 16), np.float32), half=half, norm=norm, act=abi.ACT_SILU,
                       mask_coeff=0.1, device="cpu")


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("norm", [abi.NORM_DISABLED, abi.NORM_RMS, abi.NORM_LAYER, abi.NORM_BATCH])
def test_descriptor_of_each_call(half, norm):
    b = block(half, norm)
    for call, (always, with_norm) in devblock._READS.items():
        names = always + (with_norm if norm else ())
        for change in (None, "preact", "norm", "seen"):
            if change == "preact":
                b.preact = torch.zeros_like(b.preact)
            if change == "norm":
                b.leaky = b.leaky + 0.5
            full, d = b.desc(), b._fill(call)._obj
            for n, _ in abi.SklDenseDesc._fields_[:12]:
                assert getattr(d, n) == getattr(full, n), (call, n)
            for n in abi.DESC_POINTERS:
                assert getattr(d, n) == (getattr(full, n) if n in names else None), (call, n)


def test_descriptors_are_per_thread():
    b = block(True, abi.NORM_RMS)
    got = []
    t = threading.Thread(target=lambda: got.append(b._fill("forward")._obj))
    t.start()
    t.join()
    assert got[0] is not b._fill("forward")._obj


def test_leading_dimensions_of_inputs_and_targets(monkeypatch):
    """Rows and columns are the first two dimensions, whatever follows them."""
    calls = []
    monkeypatch.setattr(abi, "call", lambda name, *args: calls.append((name, args)))
    b = block(False, abi.NORM_DISABLED)
    b.forward(torch.zeros(8, 24, 1), 8)
    b.output_error(torch.zeros(8, 16, 1), abi.LOSS_CE, abi.ACT_SOFTMAX)
    b.backward(torch.zeros(8, 24, 1), abi.train_ctx(abi.sgd(0.5), abi.sgd(0.5), 8, 1e-3), 1)
    assert [args[3:5] for _, args in calls] == [(8, 24), (8, 16), (8, 24)]
