"""Softmax column sums for few query rows, whose scores the forward keeps.

Up to 32 query rows per KV head (one row more takes the pass over K), with
and without a key split, rows that see no key, key counts around the tiles of
64 and the 1024 keys of a workgroup, and column sums with their own strides.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

import flash_attn_with_score_amd as fas
from flash_attn_with_score_amd import _native
from oracle import inputs, naive
from tests.tolerances import assert_out_close, assert_sum_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, M, N, D, causal, sm_scale)
CASES = [
    (2, 4, 4, 1, 63, 64, True, None),       # one split
    (1, 8, 2, 1, 1025, 128, True, None),    # fine split, two workgroups of columns
    (1, 8, 1, 4, 2000, 128, True, -0.1),    # 32 rows
    (1, 11, 1, 3, 700, 32, True, None),     # 33 rows: the pass over K
    (1, 7, 1, 4, 4097, 16, False, 0.3),
    (3, 2, 1, 16, 9, 64, True, None),       # 7 rows see no key
    (1, 2, 2, 32, 20, 64, True, None),      # 12 rows see no key
    (1, 2, 2, 5, 1024, 64, False, 0.0),     # uniform weights
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}M{}N{}D{}{}s{}".format(*c))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_few_rows_col_softmax(case, dtype, gpu):
    B, Hq, Hk, M, N, D, causal, scale = case
    print(f"[case] few rows {case} {dtype}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=dtype, seed=17)
    o, col = fas.attention_with_softmax_col_sum(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal,
                                                sm_scale=scale)
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=causal, sm_scale=scale,
                                  want=("out", "col_softmax"))
    assert_out_close(o, ref["out"])
    assert_sum_close(col, ref["col_softmax"], "col_softmax")


def test_few_rows_strided_sums(gpu):
    """Column sums with a stride of 3 and gaps that stay as they were."""
    B, Hq, Hk, M, N, D = 2, 4, 2, 2, 700, 64
    print("[case] few rows, strided sums", flush=True)
    lib = _native.load()
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=torch.float16, seed=4)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    o = torch.empty_like(qd)
    args = _native.make_args(qd, kd, vd, o, True, D ** -0.5)
    nbytes = lib.fas_workspace_bytes(_native.VARIANT_SOFTMAX_COL_SUM, ctypes.byref(args), 0)
    ws = torch.full((nbytes + 256,), 0xFF, dtype=torch.uint8, device=gpu)
    buf = torch.full((B, Hk, N, 3), -7.0, device=gpu)
    rc = lib.fas_attention_with_softmax_col_sum(
        ctypes.byref(args), buf.data_ptr(), _native._I64x3(Hk * N * 3, N * 3, 3),
        ws.data_ptr() + (-ws.data_ptr()) % 256, nbytes, torch.cuda.current_stream().cuda_stream)
    _native.check(lib, rc, "fas_attention_with_softmax_col_sum")
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=True, want=("col_softmax",))
    assert_sum_close(buf[..., 0], ref["col_softmax"], "col_softmax")
    assert (buf[..., 1:] == -7.0).all()
