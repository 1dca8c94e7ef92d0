"""The C ABI's buffered cross-token softmax sum (the region's scores kept in the
caller's workspace), which the Python entry point takes for small regions only."""
from __future__ import annotations

import ctypes

import torch

from flash_attn_with_score_amd import _native

ENTRIES = {_native.VARIANT_CROSS_SOFTMAX_SUM: "fas_attention_cross_token_softmax_sum",
           _native.VARIANT_CROSS_SOFTMAX_SUM_BUFFERED:
               "fas_attention_cross_token_softmax_sum_buffered"}


def cross_softmax_sum(variant, q, k, v, split, causal):
    """(out, sums) of one C entry point, outputs and workspace filled with NaN."""
    lib, name = _native.load(), ENTRIES[variant]
    B, Hk, D = k.shape[0], k.shape[1], k.shape[3]
    o = torch.full_like(q, float("nan"))
    x = torch.full((B, Hk, split), float("nan"), device=q.device)
    args = _native.make_args(q, k, v, o, causal, D ** -0.5)
    nbytes = lib.fas_workspace_bytes(variant, ctypes.byref(args), split)
    ws = torch.full((nbytes + 256,), 0xFF, dtype=torch.uint8, device=q.device)
    rc = getattr(lib, name)(ctypes.byref(args), split, x.data_ptr(), _native.strides3(x),
                            ws.data_ptr() + (-ws.data_ptr()) % 256, nbytes,
                            torch.cuda.current_stream().cuda_stream)
    _native.check(lib, rc, name)
    torch.cuda.synchronize()
    return o, x


def buffered(q, k, v, split, causal):
    return cross_softmax_sum(_native.VARIANT_CROSS_SOFTMAX_SUM_BUFFERED, q, k, v, split, causal)
