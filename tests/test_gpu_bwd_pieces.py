"""dK/dV with a key block's row tiles dealt to several workgroups.

Few KV heads over long query ranges: pieces that start and end inside a
head, pieces of key blocks that few or no rows see, grouped query heads,
ragged rows and keys, and the dropout mask, against the oracle.
"""
from __future__ import annotations

import pytest
import torch

import flash_attn_with_score_amd as fas
from oracle import inputs, naive
from tests.tolerances import assert_out_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, M, N, D, causal, dropout)
CASES = [
    (1, 2, 2, 1030, 1030, 64, True, 0.0),    # 17 row tiles in 4 pieces
    (1, 1, 1, 2050, 130, 32, False, 0.0),    # 33 tiles, two key blocks, the last of 2 keys
    (1, 2, 2, 1200, 700, 64, True, 0.0),     # 500 rows see no key
    (1, 2, 2, 600, 1400, 16, True, 0.0),     # every row sees the first key blocks
    (1, 4, 1, 700, 900, 128, True, 0.0),     # four query heads: pieces across heads
    (1, 7, 1, 300, 333, 128, False, 0.0),    # seven query heads of five tiles
    (2, 6, 2, 520, 520, 64, True, 0.2),
    (1, 2, 2, 1030, 1030, 128, False, 0.2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}M{}N{}D{}{}p{}".format(*c))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_dkdv_pieces(case, dtype, gpu):
    B, Hq, Hk, M, N, D, causal, p = case
    print(f"[case] dK/dV pieces {case} {dtype}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=dtype, seed=13)
    do = torch.randn(q.shape, generator=torch.Generator("cpu").manual_seed(2)).to(dtype)
    qg, kg, vg = (t.to(gpu).requires_grad_(True) for t in (q, k, v))
    torch.cuda.manual_seed(5)
    o, _, _, seed, off = fas.attention(qg, kg, vg, causal=causal, dropout_p=p,
                                       return_log_normalizer=True, return_seed_offset=True)
    dq, dk, dv = torch.autograd.grad(o, (qg, kg, vg), do.to(gpu))
    torch.cuda.synchronize()
    drop = (p, seed, off) if p else None
    ref = naive.attention_reference(q, k, v, do, causal=causal, dropout=drop)
    for name, got in (("out", o), ("dq", dq), ("dk", dk), ("dv", dv)):
        assert_out_close(got, ref[name], name)
