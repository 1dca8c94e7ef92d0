"""The C ABI's buffered cross-token softmax sum, which keeps the region's
scores in the caller's workspace, against the recomputing entry point and the
oracle."""
from __future__ import annotations

import pytest
import torch

from flash_attn_with_score_amd import _native
from oracle import inputs, naive
from tests.buffered import cross_softmax_sum
from tests.tolerances import assert_out_close, assert_sum_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, S, D, split, causal): splits with 16-byte rows, 8-byte rows and neither
CASES = [(1, 4, 2, 300, 64, 136, True), (2, 3, 3, 257, 32, 100, False), (1, 7, 1, 200, 128, 77, True),
         (1, 2, 2, 520, 16, 513, True),
         # several units of 256 keys (64 without 8-byte rows), grouped heads, many rows
         (1, 4, 2, 1100, 64, 772, True), (2, 8, 2, 1400, 128, 1024, True),
         (1, 14, 2, 1300, 32, 600, False), (1, 6, 2, 1000, 64, 701, True),
         (3, 96, 32, 700, 64, 516, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}S{}D{}x{}{}".format(*c))
def test_buffered_entry_point(case, gpu):
    B, Hq, Hk, S, D, split, causal = case
    print(f"[case] buffered C entry point {case}", flush=True)
    q, k, v = inputs.make_qkv(B, Hq, Hk, S, S, D, dtype=torch.float16, seed=6)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    got = [cross_softmax_sum(variant, qd, kd, vd, split, causal)
           for variant in (_native.VARIANT_CROSS_SOFTMAX_SUM,
                           _native.VARIANT_CROSS_SOFTMAX_SUM_BUFFERED)]
    assert_out_close(got[1][0], got[0][0])
    assert_sum_close(got[1][1], got[0][1], "cross_softmax")
    hk = Hk - 1
    hs = list(range(hk * (Hq // Hk), Hq))
    ref = naive.reference_forward(q[:, hs], k[:, hk:], v[:, hk:], causal=causal, split=split,
                                  want=("cross_softmax",))
    assert_sum_close(got[1][1][:, hk:], ref["cross_softmax"], "cross_softmax")
