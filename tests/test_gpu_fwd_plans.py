"""Row blocks and key splits of the plain and row-sum forward at their edges.

Row sums, outputs and log-normalizers against the oracle for 128-row blocks
whose key tiles are split between wave pairs (odd tile counts, a last pair
with one tile, rows that see no key, packed query heads, two rounds of
workgroups, dropout) and for the fine key splits of few query rows.
"""
from __future__ import annotations

import pytest
import torch

import flash_attn_with_score_amd as fas
from oracle import inputs, naive
from tests.tolerances import assert_out_close, assert_sum_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, M, N, D, causal)
CASES = [
    (1, 2, 2, 640, 640, 64, True),     # 10 key tiles, 5 steps
    (1, 2, 2, 641, 705, 128, True),    # 12 tiles, the last cut; one row in the last block
    (1, 2, 2, 127, 1090, 32, False),   # 18 tiles, less than one row block
    (1, 2, 2, 129, 833, 16, False),    # 14 tiles
    (1, 2, 2, 900, 600, 64, True),     # 300 rows see no key
    (1, 6, 2, 300, 1000, 128, True),   # three packed heads
    (1, 7, 1, 131, 1300, 64, False),   # seven packed heads
    (1, 40, 40, 1024, 1024, 16, True),  # 320 row blocks: two rounds
    (1, 8, 1, 1, 300, 64, True),       # few rows: splits of two and three tiles
    (1, 4, 1, 8, 1000, 128, True),
    (2, 32, 32, 1, 257, 32, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}M{}N{}D{}{}".format(*c))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_forward_plans(case, dtype, gpu):
    B, Hq, Hk, M, N, D, causal = case
    print(f"[case] forward plan {case} {dtype}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=dtype, seed=9)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    o, row = fas.attention_with_row_sum(qd, kd, vd, causal=causal)
    o2, L, _, _, _ = fas.attention(qd, kd, vd, causal=causal, return_log_normalizer=True)
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=causal, want=("out", "row_sum"))
    assert_out_close(o, ref["out"])
    assert_sum_close(row, ref["row_sum"], "row_sum")
    assert torch.equal(o, o2)
    s = (q.float() @ k.float().repeat_interleave(Hq // Hk, 1).transpose(-1, -2)) * D ** -0.5
    if causal:
        i, j = torch.arange(M)[:, None] + N - M, torch.arange(N)[None]
        s = s.masked_fill(j > i, float("-inf"))
    want = torch.logsumexp(s, -1)
    got = L.cpu()
    assert torch.equal(torch.isinf(got), torch.isinf(want))
    ok = ~torch.isinf(want)
    # bf16 and fp16 products are exact in fp32; the sums of up to N weights
    # in fp32 (fp16: of weights rounded to 2^-11) stay within 1e-3.
    assert (got[ok] - want[ok]).abs().max().item() < 1e-3


@pytest.mark.parametrize("case", CASES[:7], ids=lambda c: "B{}H{}K{}M{}N{}D{}{}".format(*c))
def test_forward_plans_dropout(case, gpu):
    """The dropout instances take the same row blocks: same normalizer bits,
    and the oracle's output under the generator's mask."""
    B, Hq, Hk, M, N, D, causal = case
    print(f"[case] forward plan dropout {case}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=torch.float16, seed=9)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    torch.cuda.manual_seed(77)
    o, L, _, seed, off = fas.attention(qd, kd, vd, causal=causal, dropout_p=0.3,
                                       return_log_normalizer=True, return_seed_offset=True)
    _, L0, _, _, _ = fas.attention(qd, kd, vd, causal=causal, return_log_normalizer=True)
    torch.cuda.synchronize()
    ref = naive.reference_forward(q, k, v, causal=causal, want=("out",), dropout=(0.3, seed, off),
                                  drop_scale=naive.dropout_scale(0.3))
    assert_out_close(o, ref["out"])
    assert torch.equal(L, L0)
