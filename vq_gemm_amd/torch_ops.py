"""The fused VQ GEMM as torch operators, so that graphs traced by `torch.compile` / `torch.export` can hold it as one
opaque node:

    torch.ops.vq_gemm_amd.vq_linear(x, codes, codebook, bias=None) -> Tensor

`x` is fp16 [..., K], `codes` [N, K/vec] uint8/uint16, `codebook` fp16 [E, vec] or [G, E, vec],
`bias` fp16 [N] or None; the result is fp16 [..., N].  The operators are registered by the compiled extension
(`csrc/torch_ops.cpp`, loaded here): the device implementation calls the HIP library (the current stream, no
synchronisation).  The fake implementations below only propagate shapes.  There is no CPU implementation: CPU tensors
are refused.
"""
from __future__ import annotations

import torch

from . import ops as _ops

native = _ops.load_extension("vq_gemm_torch_ops")  # registers the operators; `linear` and `gated` are the layers' direct calls


def _out_shape(x: torch.Tensor, codes: torch.Tensor, codebook: torch.Tensor):
    if codes.dim() != 2 or codebook.dim() not in (2, 3) or x.dim() < 1:
        raise ValueError("vq_linear: x [..., K], codes [N, K/vec], codebook [E, vec] or [G, E, vec]")
    if codes.dtype not in (torch.uint8, torch.uint16):
        raise ValueError(f"vq_linear: codes must be uint8 or uint16, got {codes.dtype}")
    if x.shape[-1] != codes.shape[1] * codebook.shape[-1]:
        raise ValueError(f"vq_linear: x has {x.shape[-1]} features, codes x vec give {codes.shape[1] * codebook.shape[-1]}")
    return (*x.shape[:-1], codes.shape[0])


# x @ W.T (+ bias) on a code matrix [N, K/vec]
vq_linear = torch.ops.vq_gemm_amd.vq_linear
# `vq_linear` on a code matrix in the decode kernel's packed layout (`cabi.pack_codes_b`): the decode kernel only, for
# the shapes `cabi.decode_packed_supports` accepts
vq_linear_packed = torch.ops.vq_gemm_amd.vq_linear_packed
# silu(gate_up[..., :N]) * gate_up[..., N:] for fp16 gate_up [..., 2N]
silu_mul = torch.ops.vq_gemm_amd.silu_mul
# silu(x @ Wg.T) * (x @ Wu.T) in one fused VQ GEMM: `codes` [2H, K/vec] hold the gate and the up rows interleaved in
# groups of 16 (`vq_gemm_amd.quantize.interleave_gate_up`), the result is fp16 [..., H]
vq_gated_linear = torch.ops.vq_gemm_amd.vq_gated_linear


@torch.library.register_fake("vq_gemm_amd::vq_linear")
def _vq_linear_fake(x, codes, codebook, bias=None):
    return x.new_empty(_out_shape(x, codes, codebook))


@torch.library.register_fake("vq_gemm_amd::vq_linear_packed")
def _vq_linear_packed_fake(x, codes_packed, codebook, bias=None):
    return x.new_empty(_out_shape(x, codes_packed, codebook))


@torch.library.register_fake("vq_gemm_amd::silu_mul")
def _silu_mul_fake(gate_up):
    if gate_up.shape[-1] % 2 != 0:
        raise ValueError("silu_mul: expected an even last dimension")
    return gate_up.new_empty((*gate_up.shape[:-1], gate_up.shape[-1] // 2))


@torch.library.register_fake("vq_gemm_amd::vq_gated_linear")
def _vq_gated_linear_fake(x, codes, codebook, bias=None):
    shape = _out_shape(x, codes, codebook)
    return x.new_empty((*shape[:-1], shape[-1] // 2))
