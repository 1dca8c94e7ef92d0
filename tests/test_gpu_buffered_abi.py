"""The C ABI's buffered cross-token softmax sum, which keeps the region's
scores in the caller's workspace, against the recomputing entry point."""
from __future__ import annotations

import ctypes

import pytest
import torch

from flash_attn_with_score_amd import _native
from oracle import inputs
from tests.tolerances import assert_out_close, assert_sum_close

pytestmark = pytest.mark.gpu

# (B, Hq, Hk, S, D, split, causal): splits with 16-byte rows, 8-byte rows and neither
CASES = [(1, 4, 2, 300, 64, 136, True), (2, 3, 3, 257, 32, 100, False), (1, 7, 1, 200, 128, 77, True),
         (1, 2, 2, 520, 16, 513, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}S{}D{}x{}{}".format(*c))
def test_buffered_entry_point(case, gpu):
    B, Hq, Hk, S, D, split, causal = case
    print(f"[case] buffered C entry point {case}", flush=True)
    lib = _native.load()
    q, k, v = (t.to(gpu) for t in inputs.make_qkv(B, Hq, Hk, S, S, D, dtype=torch.float16, seed=6))
    stream = torch.cuda.current_stream().cuda_stream
    got = {}
    for name, variant in (("fas_attention_cross_token_softmax_sum", 6),
                          ("fas_attention_cross_token_softmax_sum_buffered", 7)):
        o, x = torch.empty_like(q), torch.full((B, Hk, split), float("nan"), device=gpu)
        args = _native.make_args(q, k, v, o, causal, D ** -0.5)
        nbytes = lib.fas_workspace_bytes(variant, ctypes.byref(args), split)
        ws = torch.full((nbytes + 256,), 0xFF, dtype=torch.uint8, device=gpu)
        rc = getattr(lib, name)(ctypes.byref(args), split, x.data_ptr(), _native.strides3(x),
                                ws.data_ptr() + (-ws.data_ptr()) % 256, nbytes, stream)
        _native.check(lib, rc, name)
        got[variant] = (o, x)
    torch.cuda.synchronize()
    assert_out_close(got[7][0], got[6][0])
    assert_sum_close(got[7][1], got[6][1], "cross_softmax")
