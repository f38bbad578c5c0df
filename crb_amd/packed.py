"""Packed low-bit linear layers for inference.

The reference stores a quantized layer as fake-quantized fp16/bf16 weights
(bigptq.py:278-280).  ``PackedLinear`` keeps the same weights exactly in
3 bits each (2-bit codes, an 8-entry value table per 128-column block
row, one salient-column bitmap per block; the format is described in
include/crbq.h) and multiplies with them directly: up to 16 tokens per call
through the packed GEMV (MFMA on weights decoded in registers), up to 768
through the packed GEMM (each decoded fragment reused for up to 128 tokens),
with bias and rounding in the same kernels, and larger batches by unpacking
into a temporary dense weight for the dense GEMM.  The second limit bounds
memory (up to 768 tokens no temporary weight is allocated); in time the dense
route wins from about 512 tokens on the larger layers.  Packed / through the
dense weight on MI355X, us: 4096 x 16384 at 256 / 512 / 768 / 1024 tokens 62 /
94, 101 / 117, 151 / 136, 177 / 159; 16384 x 4096 59 / 70, 85 / 89, 160 / 109,
169 / 128; 4096 x 4096 28 / 31, 38 / 38, 55 / 43, 59 / 49; 1024 x 4096 18 / 31,
20 / 31, 26 / 31, 28 / 31; 768 x 768 15 / 31, 15 / 31, 16 / 31, 16 / 31.
"""
from __future__ import annotations

from operator import itemgetter

import torch
import torch.autograd.forward_ad as fwad
import torch.nn as nn
import torch.nn.functional as F

from . import kernels
from ._lib import LINEAR_MAX_EX

GEMV_MAX_TOKENS = 16
GEMM_MAX_TOKENS = 768
_parts = itemgetter("codes", "lut", "sal", "bias", "ex_idx")
_wrapped = torch._C._functorch.is_functorch_wrapped_tensor
_PLAIN = frozenset((torch.Tensor, nn.Parameter))


def _plain(b: torch.Tensor) -> bool:
    """Whether a kernel may read b's memory in the place of torch's add: no
    gradient, no forward-mode tangent, no torch.func wrapper, no subclass, no
    negated view."""
    return (type(b) in _PLAIN and not b.requires_grad and not b.is_neg() and not _wrapped(b)
            and (fwad._current_level < 0 or fwad.unpack_dual(b).tangent is None))


class PackedLinear(nn.Module):
    """nn.Linear with packed weights (in_features = C, out_features = R).
    Buffers: codes, lut, sal (the 3-bit form) and ex_idx, ex_val, ex_delta
    (the rare weights outside their group's table, usually none)."""

    def __init__(self, codes, lut, sal, in_features, bias=None, ex=None):
        super().__init__()
        self.in_features = int(in_features)
        self.out_features = codes.shape[0]
        self.register_buffer("codes", codes)
        self.register_buffer("lut", lut)
        self.register_buffer("sal", sal)
        if ex is None:
            dev = codes.device
            ex = kernels.PackedEx(torch.empty(0, dtype=torch.int64, device=dev),
                                  torch.empty(0, dtype=lut.dtype, device=dev),
                                  torch.empty(0, dtype=torch.float32, device=dev))
        self.register_buffer("ex_idx", ex.idx)
        self.register_buffer("ex_val", ex.val)
        self.register_buffer("ex_delta", ex.delta)
        self.register_buffer("bias", bias)

    @property
    def ex(self) -> kernels.PackedEx:
        return kernels.PackedEx(self.ex_idx, self.ex_val, self.ex_delta)

    @classmethod
    def from_linear(cls, layer: nn.Linear, masks: torch.Tensor) -> "PackedLinear":
        """Pack a quantized nn.Linear given the mask codes its block loop used."""
        codes, lut, sal, ex = kernels.pack(layer.weight.data, masks)
        b = layer.bias.data.clone() if layer.bias is not None else None
        return cls(codes, lut, sal, layer.in_features, b, ex)

    def weight(self) -> torch.Tensor:
        """The dense quantized weight (bit-identical to what was packed)."""
        return kernels.unpack(self.codes, self.lut, self.sal, self.in_features, self.ex)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        shape = x.shape
        x2 = x.reshape(-1, self.in_features)
        try:                         # one token's call is host time: no attribute look-ups
            codes, lut, sal, bias, ex_idx = _parts(self._buffers)
        except KeyError:             # one was assigned as a Parameter, or parametrized
            codes, lut, sal, bias, ex_idx = (self.codes, self.lut, self.sal, self.bias,
                                             self.ex_idx)
        n_ex = ex_idx.numel()
        # product, exceptions, bias and rounding in one kernel: activations and
        # bias in the weights' dtype, few exceptions, a plain [R] bias (one that
        # broadcasts or that torch has to see is added on its own)
        if (x2.shape[0] <= GEMM_MAX_TOKENS and x.dtype == lut.dtype and n_ex <= LINEAR_MAX_EX
                and (bias is None or (bias.dtype == x.dtype and bias.is_contiguous()
                                      and bias.shape == (self.out_features,)
                                      and _plain(bias)))):
            y = kernels.linear_packed(codes, lut, sal, self.in_features, x2, bias,
                                      self.ex if n_ex else None)
        elif x2.shape[0] <= GEMM_MAX_TOKENS:
            mm = kernels.gemv_packed if x2.shape[0] <= GEMV_MAX_TOKENS else kernels.gemm_packed
            y = mm(codes, lut, sal, self.in_features, x2, self.ex)
            y = y.to(x.dtype)
            if bias is not None:
                y = y + bias
        else:
            y = F.linear(x2.to(lut.dtype), self.weight(), bias)
        return y.reshape(*shape[:-1], self.out_features)

    def packed_bytes(self) -> int:
        return sum(t.numel() * t.element_size()
                   for t in (self.codes, self.lut, self.sal, self.ex_idx, self.ex_val,
                             self.ex_delta))


def replace_linears(module: nn.Module, packed: dict) -> None:
    """Swap named nn.Linear submodules of module for their PackedLinear."""
    for name, pl in packed.items():
        parent = module
        parts = name.split(".")
        for p in parts[:-1]:
            parent = getattr(parent, p)
        setattr(parent, parts[-1], pl)
