"""Cross-token softmax-weight sums, and the buffered variant's entry point.

Drop-ins for the reference's attention_cross_token_softmax_sum.py:735-863
(attention_cross_token_softmax_sum, fused two-pass kernel :24-268) and
:639-732 (attention_cross_token_softmax_sum_buffered, kernel :434-636).
"""
from __future__ import annotations


import torch

from . import _common, _native

__all__ = ["attention_cross_token_softmax_sum", "attention_cross_token_softmax_sum_buffered"]

# The buffered variant keeps the region's scores only for at most
# BUFFERED_ROWS query rows past the split over at most BUFFERED_KEYS keys, where
# a column pass of its own costs more than the little it writes (us, buffered /
# recomputed, D128: B4 H4 S296 split 250 23.4 / 24.6, split 232 20.6 / 24.5; B1
# H12 S704 split 640 34.3 / 32.0; B1 H32 S2048 split 2000 79.5 / 63.0).
BUFFERED_ROWS, BUFFERED_KEYS = 64, 512


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
    the region (queries >= split, keys < split) is faster than writing and reading even 2 bytes per score of it
    (fas_attention_cross_token_softmax_sum_buffered: B1 H32/8 S16384 split
    12288 D128 2.94 against 2.35 ms, B1 H32 S4096 split 3072 231 against 190
    us, split 3001 560 against 193 us, B1 H4 S1664 split 283 D32 151 against
    53 us), is exact to fp32 instead of fp16 exponents, and needs no region,
    so this entry point recomputes too, but for the few rows of
    BUFFERED_ROWS.
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
    if M - split <= BUFFERED_ROWS and N <= BUFFERED_KEYS:
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
