"""Softmax column sums whose row steps are dealt to several workgroups.

Few heads over long query ranges: pieces that start and end inside a head,
key blocks few rows see, a cross-token split, dropout; against the oracle, and
the same bits on a second call (the pieces are added in order).
"""
from __future__ import annotations

import pytest
import torch

import flash_attn_with_score_amd as fas
from oracle import inputs, naive
from tests.tolerances import assert_sum_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, M, N, D, causal, split)
CASES = [
    (1, 2, 2, 1300, 1300, 64, True, 0),    # 11 row steps, 3 mirror pairs
    (1, 1, 1, 2000, 100, 128, False, 0),   # one key block, 16 steps
    (1, 3, 1, 700, 900, 32, True, 0),      # three heads of 6 steps
    (1, 2, 1, 1100, 600, 16, True, 0),     # 500 rows see no key
    (1, 2, 2, 1664, 1664, 32, False, 283),
    (1, 4, 2, 1200, 1200, 64, True, 700),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}M{}N{}D{}{}x{}".format(*c))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_column_row_pieces(case, dtype, gpu):
    B, Hq, Hk, M, N, D, causal, split = case
    print(f"[case] column row pieces {case} {dtype}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=dtype, seed=19)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    if split:
        call = lambda: fas.attention_cross_token_softmax_sum(qd, kd, vd, split, causal=causal)[1]  # noqa: E731
        want = "cross_softmax"
    else:
        call = lambda: fas.attention_with_softmax_col_sum(qd, kd, vd, causal=causal)[1]  # noqa: E731
        want = "col_softmax"
    col = call()
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=causal, split=split or None, want=(want,))
    assert_sum_close(col, ref[want], want)
    assert torch.equal(col, call())


def test_column_row_pieces_dropout(gpu):
    B, H, S, D, p = 1, 2, 1300, 64, 0.25
    print("[case] column row pieces, dropout", flush=True)
    q, k, v = inputs.make_qkv(B, H, H, S, S, D, dtype=torch.float16, seed=19)
    torch.cuda.manual_seed(3)
    _, col = fas.attention_with_softmax_col_sum(q.to(gpu), k.to(gpu), v.to(gpu), causal=True,
                                                dropout_p=p)
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=True, want=("col_softmax",), dropout=(p, 3, 0),
                                  drop_col_softmax=True)
    assert_sum_close(col, ref["col_softmax"], "col_softmax")
