"""Device-side DenseBlock state for driving the C ABI from Python.

`DeviceBlock` owns one block's device buffers (torch tensors used purely as
device memory) laid out exactly as `skl_dense_desc` expects, initialised the
way src/mlp.rs:45-110 / 377-421 initialises a block: W from the caller, bias
and norm bias 0, norm weight 1, moments 0, caches 0, mask 1, and for fp16
blocks fp32 masters.  Every hot-path step is one C-ABI call.
"""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import torch

from . import abi

T_FIELDS = ("w", "b", "norm_w", "norm_b", "out", "predrop", "preact", "centered", "prenorm", "norm_rstd", "mask")
F32_FIELDS = ("master_w", "master_b", "master_norm_w", "master_norm_b",
              "dv_w", "dv_b", "dm_w", "dm_b", "dv_norm_w", "dv_norm_b", "dm_norm_w", "dm_norm_b",
              "grad", "d_prenorm", "d_norm_w", "d_norm_b")


# The descriptor pointers each call reads (src/io/device/ffn_device.rs), without a norm and
# those that come with one.  A descriptor of 28 tensors costs more to fill than the launch it
# describes (3.4 us; 9.2 us for a whole forward call), so each call fills its own few.
_NORM_CACHES = ("norm_w", "norm_b", "centered", "prenorm", "norm_rstd")
_ERROR = ("w", "preact", "grad", "d_prenorm", "d_prenorm_h")
_ERROR_NORM = _NORM_CACHES + ("d_norm_w", "d_norm_b", "master_norm_w")
_UPDATE = ("w", "b", "master_w", "master_b", "dv_w", "dm_w", "dv_b", "dm_b", "grad", "d_prenorm", "d_prenorm_h")
_UPDATE_NORM = _ERROR_NORM + ("master_norm_b", "dv_norm_w", "dm_norm_w", "dv_norm_b", "dm_norm_b")
_READS = {
    "forward": (("w", "b", "out", "predrop", "preact", "mask"), _NORM_CACHES),
    "output_error": (_ERROR + ("out",), _ERROR_NORM),
    "error": (_ERROR + ("predrop", "mask"), _ERROR_NORM),
    "input_grad": (("w", "d_prenorm", "d_prenorm_h"), ()),
    "above": (("w", "d_prenorm", "d_prenorm_h"), ()),
    "update": (_UPDATE, _UPDATE_NORM),
    "hidden": (_UPDATE + ("predrop", "preact", "mask"), _UPDATE_NORM),
}
_SCALARS = tuple(n for n, _ in abi.SklDenseDesc._fields_[:11])
_PTR_AT = {n: getattr(abi.SklDenseDesc, n).offset // 8 for n in abi.DESC_POINTERS}


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


class DeviceBlock:
    def __init__(self, ctx: abi.Context, inputs: int, outputs: int, max_batch: int, w: np.ndarray, *,
                 half: bool = False, norm: int = 0, act: int = 0, leaky: float = 0.0, mask_coeff: float = 0.0,
                 regularisation: int = 0, regu_coeff: float = 0.0, is_training: bool = True,
                 master_w: np.ndarray | None = None, b: np.ndarray | None = None, device: str = "cuda"):
        self.ctx = ctx
        self.half = half
        self.inputs, self.outputs, self.max_batch = inputs, outputs, max_batch
        self.norm, self.act, self.leaky, self.mask_coeff = norm, act, leaky, mask_coeff
        self.regularisation, self.regu_coeff = regularisation, regu_coeff
        self.is_training = is_training
        K, N, M = inputs, outputs, max_batch
        T = torch.float16 if half else torch.float32
        self.tdtype = T
        dev = torch.device(device)

        def up(a, dt):
            return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(device=dev, dtype=dt).contiguous()

        def zeros(shape, dt):
            return torch.zeros(shape, device=dev, dtype=dt)

        w = np.asarray(w, np.float32).reshape(K, N)
        self.w = up(w, T)
        self.b = zeros((1, N), T) if b is None else up(np.asarray(b, np.float32).reshape(1, N), T)
        self.norm_w = torch.ones((1, N), device=dev, dtype=T)
        self.norm_b = zeros((1, N), T)
        if half:
            self.master_w = up(master_w.reshape(K, N) if master_w is not None else self.w.float().cpu().numpy(),
                               torch.float32)
            self.master_b = self.b.float().clone()
            self.master_norm_w = torch.ones((1, N), device=dev, dtype=torch.float32)
            self.master_norm_b = zeros((1, N), torch.float32)
        else:
            self.master_w = self.master_b = self.master_norm_w = self.master_norm_b = None
        for n, shape in (("dv_w", (K, N)), ("dm_w", (K, N)), ("dv_b", (1, N)), ("dm_b", (1, N)),
                         ("dv_norm_w", (1, N)), ("dv_norm_b", (1, N)), ("dm_norm_w", (1, N)),
                         ("dm_norm_b", (1, N))):
            setattr(self, n, zeros(shape, torch.float32) if is_training else None)
        for n in ("out", "predrop", "preact", "centered", "prenorm"):
            setattr(self, n, zeros((M, N), T))
        self.norm_rstd = zeros((max(M, N),), T)
        self.mask = torch.ones((M, N), device=dev, dtype=T)
        for n in ("grad", "d_prenorm", "d_norm_w", "d_norm_b"):
            setattr(self, n, zeros((M, N), torch.float32) if is_training else None)
        self.d_prenorm_h = zeros((M, N), torch.float16) if (half and is_training) else None
        self._desc = None
        self._local = threading.local()   # _fill's descriptors, one set per thread

    # -- descriptor -----------------------------------------------------------------
    def desc(self) -> abi.SklDenseDesc:
        d = abi.SklDenseDesc()
        d.dtype = abi.F16 if self.half else abi.F32
        d.inputs, d.outputs, d.max_batch = self.inputs, self.outputs, self.max_batch
        d.norm, d.act, d.leaky, d.mask_coeff = self.norm, self.act, self.leaky, self.mask_coeff
        d.regularisation, d.regu_coeff = self.regularisation, self.regu_coeff
        d.is_training = int(self.is_training)
        for n in T_FIELDS + F32_FIELDS + ("d_prenorm_h",):
            setattr(d, n, _ptr(getattr(self, n)))
        self._desc = d
        return d

    def _fill(self, call: str):
        """Reference to this call's own descriptor with its pointers read from the tensors as
        they are now; the pointers it does not read stay null."""
        key = (self.half, self.inputs, self.outputs, self.max_batch, self.norm, self.act, self.leaky, self.mask_coeff,
               self.regularisation, self.regu_coeff, self.is_training)
        descs = self._local.__dict__
        kept = descs.get(call)
        if kept is None or kept[0] != key:
            d = abi.SklDenseDesc()
            for n, v in zip(_SCALARS, (abi.F16 if self.half else abi.F32,) + key[1:10] + (int(self.is_training),)):
                setattr(d, n, v)
            names, with_norm = _READS[call]
            at = tuple((n, _PTR_AT[n]) for n in (names + with_norm if self.norm else names))
            kept = descs[call] = (key, C.byref(d), memoryview(d).cast("B").cast("Q"), at)
        _, ref, words, at = kept
        tensors = self.__dict__
        for n, i in at:
            t = tensors[n]
            words[i] = 0 if t is None else t.data_ptr()
        return ref

    # -- hot-path steps ------------------------------------------------------------------
    def forward(self, x: torch.Tensor, batch: int, use_dropout: bool = False, seed: int = 0):
        rows, cols = x.shape[0], x.shape[1]
        abi.call("skl_dense_forward", self.ctx.h, self._fill("forward"), x.data_ptr(), rows, cols, batch,
                 int(use_dropout), seed & 0xFFFFFFFF)
        return self.out

    def output_error(self, target: torch.Tensor, loss: int, act: int, leaky: float = 0.0):
        rows, cols = target.shape[0], target.shape[1]
        abi.call("skl_dense_output_error", self.ctx.h, self._fill("output_error"), target.data_ptr(), rows, cols, loss,
                 act, leaky)

    def hidden_error(self, nxt: "DeviceBlock", batch: int):
        abi.call("skl_dense_hidden_error", self.ctx.h, self._fill("hidden"), nxt._fill("above"), batch)

    def backward(self, x: torch.Tensor, tc: abi.SklTrainCtx, step: int):
        rows, cols = x.shape[0], x.shape[1]
        abi.call("skl_dense_backward", self.ctx.h, self._fill("update"), x.data_ptr(), rows, cols, C.byref(tc), step)

    def backward_hidden(self, nxt: "DeviceBlock", x: torch.Tensor, tc: abi.SklTrainCtx, step: int):
        rows, cols = x.shape[0], x.shape[1]
        abi.call("skl_dense_backward_hidden", self.ctx.h, self._fill("hidden"), nxt._fill("above"), x.data_ptr(), rows,
                 cols, C.byref(tc), step)

    def error_from_sum(self, s: torch.Tensor, batch: int):
        assert s.dtype == torch.float32 and s.is_contiguous()
        abi.call("skl_dense_error_from_sum", self.ctx.h, self._fill("error"), s.data_ptr(), batch)

    def error_from_sum_noalloc(self, s: torch.Tensor, batch: int):
        assert s.dtype == torch.float32 and s.is_contiguous()
        abi.call("skl_dense_error_from_sum_noalloc", self.ctx.h, self._fill("error"), s.data_ptr(), batch)

    def input_grad(self, batch: int, out: torch.Tensor | None = None) -> torch.Tensor:
        if out is None:
            out = torch.empty((batch, self.inputs), device=self.w.device, dtype=torch.float32)
        abi.call("skl_dense_input_grad", self.ctx.h, self._fill("input_grad"), batch, out.data_ptr())
        return out

    # -- host views ----------------------------------------------------------------------
    def get(self, name: str) -> np.ndarray | None:
        t = getattr(self, name)
        return None if t is None else t.float().cpu().numpy()

    def snapshot(self) -> dict:
        return {n: self.get(n) for n in T_FIELDS + F32_FIELDS}
