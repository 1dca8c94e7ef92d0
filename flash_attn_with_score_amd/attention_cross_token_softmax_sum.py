"""Cross-token softmax-weight sums, and the buffered variant's entry point.

Drop-ins for the reference's attention_cross_token_softmax_sum.py:735-863
(attention_cross_token_softmax_sum, fused two-pass kernel :24-268) and
:639-732 (attention_cross_token_softmax_sum_buffered, kernel :434-636).
"""
from __future__ import annotations


import torch

from . import _common, _native

__all__ = ["attention_cross_token_softmax_sum", "attention_cross_token_softmax_sum_buffered"]

# The buffered variant keeps the region's scores only where that is faster than
# a second pass over K: at most BUFFERED_ROWS query rows past the split over at
# most BUFFERED_KEYS keys whose region rows start on 16 bytes, or at any split
# over at most BUFFERED_SHORT keys.  Time kept / recomputed, mean over six head
# counts and D = 32, 64, 128 (fp16, causal), 64 rows: S 200 0.96, 296 0.95, 384
# 0.90, 448 1.00, 512 1.04; 8 rows 0.83, 0.82, 0.83, 0.92, 0.97; 128 rows 1.02
# to 1.09; splits that are no multiple of 8, 33 rows: S 136 0.91, 200 1.08, 296
# 1.10, 384 1.14, 448 1.32, 512 1.45.
BUFFERED_ROWS, BUFFERED_KEYS, BUFFERED_SHORT = 64, 448, 160


def _keeps_region(M: int, N: int, split: int) -> bool:
    keys = BUFFERED_KEYS if split % 8 == 0 else BUFFERED_SHORT
    return M - split <= BUFFERED_ROWS and N <= keys


def attention_cross_token_softmax_sum_buffered(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    split: int,
    causal: bool = False,
    sm_scale: float = None,
    dropout_p: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Same result as attention_cross_token_softmax_sum.

    The reference's pass 1 stores the raw scores, B * Hq * M * N * 4 bytes
    (:704-705), and its pass 2 reloads them.  On MI355X recomputing q . k for
    the region (queries >= split, keys < split) is faster than writing and
    reading even 2 bytes per score of it, is exact to fp32 instead of fp16
    exponents, and needs no region, so this entry point recomputes too, but for
    the small regions of _keeps_region
    (fas_attention_cross_token_softmax_sum_buffered).
    """
    Dq, Dk, Dv = q.shape[-1], k.shape[-1], v.shape[-1]
    assert Dq == Dk == Dv, "Q, K, V must have the same head_dim"
    assert Dk in {16, 32, 64, 128}

    B, H, M, D = q.shape
    N = k.shape[2]
    Hk = k.shape[1]
    Hv = v.shape[1]
    assert Hk == Hv, "K and V must have the same number of heads"
    assert H % Hk == 0, "num_heads_q must be divisible by num_heads_k"

    assert 0 < split <= N, f"Split position must be in valid range (0, {N}]"

    _common.check_device_inputs(q, k, v, dropout_p)
    p = _common.finish_problem(q, k, v, sm_scale)
    output = _common.new_output(p.q)
    cross = torch.empty((B, Hk, split), device=q.device, dtype=torch.float32)
    # The reference's buffered kernel ignores dropout_p and draws no seed.
    args = _native.pack_args(p.q, p.k, p.v, output, causal, p.sm_scale)
    variant, entry = _native.VARIANT_CROSS_SOFTMAX_SUM, "fas_attention_cross_token_softmax_sum"
    if _keeps_region(M, N, split):
        variant, entry = _native.VARIANT_CROSS_SOFTMAX_SUM_BUFFERED, entry + "_buffered"
    ws_ptr, ws_bytes, ws = _common.workspace(variant, args, split, q.device)
    _common.call(entry, p.q, args, int(split), cross.data_ptr(), _native.pack_strides(cross), ws_ptr,
                 ws_bytes)
    return output, cross


def attention_cross_token_softmax_sum(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    split: int,
    causal: bool = False,
    sm_scale: float = None,
    dropout_p: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Returns (output, cross_token_softmax_sum (B, Hk, split) fp32) with
    sum[b, hk, j] = sum over queries i in [split, M) and the query heads of
    group hk of exp(s_ij - m_i) / (l_i + 1e-12), for keys j < split
    (attention_cross_token_softmax_sum.py:236-268)."""
    Dq, Dk, Dv = q.shape[-1], k.shape[-1], v.shape[-1]
    assert Dq == Dk == Dv, "Q, K, V must have the same head_dim"
    assert Dk in {16, 32, 64, 128}

    B, H, M, D = q.shape
    N = k.shape[2]
    Hk = k.shape[1]
    assert Hk == v.shape[1]
    assert H % Hk == 0

    assert 0 < split <= N, f"Split position must be in valid range (0, {N}]"

    _common.check_device_inputs(q, k, v, dropout_p)
    p = _common.finish_problem(q, k, v, sm_scale)
    output = _common.new_output(p.q)
    cross = torch.empty((B, Hk, split), device=q.device, dtype=torch.float32)
    args = _native.pack_args(p.q, p.k, p.v, output, causal, p.sm_scale,
                             _common.draw_dropout(p.q, p.k, dropout_p))
    ws_ptr, ws_bytes, ws = _common.workspace(_native.VARIANT_CROSS_SOFTMAX_SUM, args, split,
                                             q.device)
    _common.call("fas_attention_cross_token_softmax_sum", p.q, args, int(split),
                 cross.data_ptr(), _native.pack_strides(cross), ws_ptr, ws_bytes)
    return output, cross
