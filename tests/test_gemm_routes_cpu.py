"""The GEMM planner without a GPU: the kernel it gives to sizes that must not reach another one."""
from __future__ import annotations

import ctypes as C
import os

import pytest

from soklyn_amd import abi

F32, F16 = 0, 1
FWD, DX, DW, HID = 0, 1, 2, 3


@pytest.fixture(scope="module")
def route():
    if not os.path.exists(abi.LIB_PATH):
        pytest.skip("libsoklyn_hip.so not built")
    f = C.CDLL(abi.LIB_PATH).skl_diag_gemm_route
    f.restype, f.argtypes = C.c_char_p, [C.c_uint32] * 5
    return lambda *a: f(*a).decode()


# dW of a narrow layer whose input passes 2 GiB: the K-splitting kernel's 32-bit offsets end there
# in one slice, and 128-column tiles would be 7/8 padding read element by element
@pytest.mark.parametrize("dtype", [F16, F32])
@pytest.mark.parametrize("inputs,outputs,batch", [(16384, 10, 65536), (16384, 10, 131072), (8192, 16, 262144),
                                                  (4096, 10, 2000000), (100000, 1, 20000)])
def test_narrow_dw_over_a_very_large_input(route, dtype, inputs, outputs, batch):
    assert route(dtype, DW, inputs, outputs, batch).split(":")[0] in ("skinny", "wave")


# ... and where its stream over X is slower: rows at odd pitches, from 64 MB on
@pytest.mark.parametrize("dtype,inputs,outputs,batch", [(F16, 12559, 6, 35630), (F16, 29256, 7, 18807),
                                                        (F32, 5038, 11, 93006), (F32, 11029, 2, 31645)])
def test_narrow_dw_streams_large_inputs_of_odd_pitch(route, dtype, inputs, outputs, batch):
    assert route(dtype, DW, inputs, outputs, batch).startswith("skinny")


@pytest.mark.parametrize("dtype", [F16, F32])
@pytest.mark.parametrize("inputs,outputs,batch", [(2048, 10, 16384), (784, 10, 64), (512, 16, 1024), (1, 1, 1)])
def test_narrow_dw_of_ordinary_sizes_takes_one_launch_or_few_slices(route, dtype, inputs, outputs, batch):
    assert route(dtype, DW, inputs, outputs, batch).startswith("wave")


# calls that routes newer than direct-to-LDS tiles (padded copies) and register-staged ones run
# slower, measured with each kernel forced (1.2-1.6x): output M x N over K
@pytest.mark.parametrize("dtype,op,M,N,K,kernel", [
    (F16, DW, 2304, 1984, 6741, "dma"), (F16, DW, 2560, 528, 13216, "dma"), (F16, DW, 3008, 3408, 6202, "staged"),
    (F32, DW, 1024, 1024, 65536, "staged"), (F32, FWD, 936, 2496, 44, "staged"), (F32, DX, 3153, 512, 192, "staged"),
    (F16, HID, 65536, 1024, 1000, "dma"), (F16, HID, 16384, 1024, 1000, "dma"), (F16, HID, 16469, 272, 55, "staged")])
def test_calls_that_the_newer_routes_slow_down_keep_theirs(route, dtype, op, M, N, K, kernel):
    assert route(dtype, op, M, N, K).split(":")[0] == kernel


# ... and that they are ahead of by 1.5x and more
@pytest.mark.parametrize("dtype,op,M,N,K,kernel", [
    (F16, FWD, 16, 4096, 4096, "wave"), (F16, FWD, 512, 2048, 2048, "wave"), (F32, FWD, 500, 1531, 777, "wave"),
    (F16, DW, 2048, 2048, 512, "wave"), (F16, DX, 2048, 1024, 1024, "wave"), (F16, HID, 512, 2048, 2048, "wave"),
    (F16, FWD, 35940, 3072, 256, "dma128")])
def test_calls_that_the_newer_routes_speed_up_take_them(route, dtype, op, M, N, K, kernel):
    assert route(dtype, op, M, N, K).split(":")[0] == kernel
