"""Score rows that do not start on 64-byte boundaries.

Each case writes the scores through the C ABI into the middle of a buffer
filled with a sentinel, with a row pitch of its own: every score must match
the oracle, and the gaps between rows and the space around the matrix must
keep the sentinel.  The shapes take each writer: key-split 64- and 128-row
blocks, 256-row blocks, packed query heads, dropout, and the scores-only
kernels (few and many query rows, behind the key-split forward).
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from flash_attn_with_score_amd import _native
from oracle import inputs, naive
from tests.tolerances import assert_out_close, assert_scores_close

pytestmark = pytest.mark.gpu

SENTINEL = 0x5A5A
# (B, Hq, Hk, M, N, D, causal, pitch - N, first element)
CASES = [
    (1, 4, 4, 130, 77, 64, True, 0, 0),       # 64-row blocks, N % 8 = 5
    (1, 4, 4, 65, 201, 128, False, 3, 1),     # odd pitch, odd first element
    (1, 2, 2, 64, 64, 32, True, 1, 0),        # whole tile, unaligned pitch
    (1, 3, 3, 70, 72, 16, False, 0, 8),       # 16-byte rows
    (1, 3, 3, 70, 96, 64, True, 0, 32),       # 64-byte rows
    (1, 3, 3, 70, 90, 64, True, 6, 32),       # 64-byte rows, N % 8 = 2
    (1, 130, 130, 100, 75, 16, False, 0, 0),  # 128-row blocks, one round
    (1, 64, 64, 520, 1031, 16, True, 0, 3),   # 128-row blocks, two rounds
    (1, 300, 300, 33, 67, 16, False, 0, 0),   # 256-row blocks
    (1, 300, 300, 70, 70, 32, True, 2, 5),    # 256-row blocks, causal zeros
    (1, 8, 2, 90, 131, 64, True, 0, 0),       # grouped heads one by one
    (40, 8, 2, 33, 67, 16, True, 0, 0),       # 256-row blocks of four packed heads
    (1, 7, 1, 66, 129, 64, True, 4, 2),       # seven heads, unpacked writer
    (1, 2, 2, 1, 7, 64, True, 0, 1),          # less than one 16-byte unit
    (1, 2, 2, 40, 2049, 64, True, 0, 0),      # key split, resident-Q scores
    (2, 4, 2, 20, 4100, 128, True, 1, 0),     # the same over two packed heads
    (1, 2, 2, 7, 2049, 64, True, 0, 1),       # few query rows: scores from the forward
    (2, 4, 2, 16, 4100, 128, True, 1, 0),     # the same, 32 rows of two packed heads
    (1, 3, 1, 1, 3007, 32, False, 0, 0),
    (1, 2, 2, 700, 3001, 32, True, 0, 0),     # key split, K-resident scores
    (64, 32, 1, 2, 2049, 16, True, 0, 0),     # 32 heads of a KV head, packed by eight
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "B{}H{}K{}M{}N{}D{}{}p{}o{}".format(*c))
@pytest.mark.parametrize("dropout", [0.0, 0.2])
def test_unaligned_score_rows(case, dropout, gpu):
    B, Hq, Hk, M, N, D, causal, gap, first = case
    print(f"[case] score rows {case} dropout={dropout}", flush=True)
    lib = _native.load()
    q, k, v = inputs.make_qkv(B, Hq, Hk, M, N, D, dtype=torch.float16, seed=5)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    o = torch.full_like(qd, float("nan"))
    drop = (dropout, 11, 4) if dropout else None
    args = _native.make_args(qd, kd, vd, o, causal, D ** -0.5, drop)
    nbytes = lib.fas_workspace_bytes(_native.VARIANT_SCORES, ctypes.byref(args), 0)
    ws = torch.empty(nbytes + 256, dtype=torch.uint8, device=gpu)
    wptr = ws.data_ptr() + (-ws.data_ptr()) % 256
    pitch, lead = N + gap, 128 + first
    rows = B * Hq * M
    buf = torch.full((lead + rows * pitch + 256,), SENTINEL, dtype=torch.int16, device=gpu)
    st = _native._I64x4(Hq * M * pitch, M * pitch, pitch, 1)
    rc = lib.fas_attention_with_scores(ctypes.byref(args), buf.data_ptr() + 2 * lead, st, wptr,
                                       nbytes, torch.cuda.current_stream().cuda_stream)
    _native.check(lib, rc, "fas_attention_with_scores")
    torch.cuda.synchronize()
    body = buf[lead:lead + rows * pitch].view(rows, pitch)
    assert (buf[:lead] == SENTINEL).all() and (buf[lead + rows * pitch:] == SENTINEL).all()
    assert (body[:, N:] == SENTINEL).all()
    got = body[:, :N].contiguous().view(torch.float16).view(B, Hq, M, N)
    heads = sorted({0, 1, Hq // 2, Hq - 1})
    ref = naive.reference_forward(q, k, v, causal=causal, want=("out", "scores"), heads=heads)
    assert_scores_close(got[:, heads], ref["scores"][:, heads])
    assert torch.isfinite(got.float()).all()
    if not dropout:
        assert_out_close(o[:, heads], ref["out"][:, heads])


# (Hq, Hk, M, N, D, causal): scores from the forward (few rows), the key-split
# route, and the fused writer with 64-, 128- and 256-row blocks; unaligned rows.
INF_CASES = [(4, 4, 3, 2048, 64, True), (8, 2, 8, 2050, 128, True), (4, 4, 2, 4096, 128, False),
             (2, 2, 40, 4096, 64, True), (2, 2, 100, 200, 128, True), (2, 2, 70, 133, 64, True),
             (130, 130, 100, 128, 16, True), (300, 300, 33, 96, 32, True)]


@pytest.mark.parametrize("case", INF_CASES, ids=lambda c: "H{}K{}M{}N{}D{}{}".format(*c))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_visible_infinite_scores_stay(case, dtype, gpu):
    """Keys of -inf and +inf scores (an infinite key element against q > 0):
    0 where the causal mask hides them, and as they are wherever it does not,
    in the diagonal's tile and in the last, partial tile too."""
    import flash_attn_with_score_amd as fas

    H, Hk, M, N, D, causal = case
    print(f"[case] infinite scores {case} {dtype}", flush=True)
    q, k, v = inputs.make_qkv(1, H, Hk, M, N, D, dtype=dtype, seed=8)
    q[..., 0] = q[..., 0].abs() + 0.5
    off = N - M
    for key, sign in ((5, -1), (64, 1), (off // 2, -1), (off, -1), (off + M // 2, -1), (N - 1, -1)):
        k[:, :, key, 0] = sign * float("inf")
    _, s = fas.attention_with_scores(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal)
    torch.cuda.synchronize()
    # Infinite products and finite ones add up to the same infinity in any order.
    heads = sorted({0, 1, H - 1})
    want = torch.matmul(q[:, heads].float(),
                        k[:, [h // (H // Hk) for h in heads]].float().transpose(-1, -2)) * D ** -0.5
    if causal:
        i, j = torch.arange(M)[:, None] + off, torch.arange(N)[None]
        want = want.masked_fill(j > i, 0.0)
    got = s[:, heads].float().cpu()
    inf = torch.isinf(want)
    assert inf.any() and torch.equal(got[inf], want[inf])
    assert_scores_close(s[:, heads].cpu().masked_fill(inf, 0.0), want.masked_fill(inf, 0.0))


# (B, Hq, Hk, N, D): the fused writer, the forward's own scores, the resident-Q
# kernel behind a key split, and (scores alone) the K-resident kernel.
ONE_ROW = [(1, 4, 4, 256, 64), (2, 2, 1, 2048, 32), (64, 64, 1, 4096, 16)]


@pytest.mark.parametrize("case", ONE_ROW, ids=lambda c: "B{}H{}K{}N{}D{}".format(*c))
@pytest.mark.parametrize("row_stride", [0, 32])
@pytest.mark.parametrize("alone", [False, True], ids=["attention", "alone"])
def test_one_row_any_row_stride(case, row_stride, alone, gpu):
    """M = 1: the row stride has no meaning, also below N."""
    B, Hq, Hk, N, D = case
    print(f"[case] one row {case} stride {row_stride} alone={alone}", flush=True)
    lib = _native.load()
    q, k, v = inputs.make_qkv(B, Hq, Hk, 1, N, D, dtype=torch.float16, seed=5)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    args = _native.make_args(qd, kd, vd, torch.empty_like(qd), True, D ** -0.5)
    nbytes = lib.fas_workspace_bytes(_native.VARIANT_SCORES, ctypes.byref(args), 0)
    ws = torch.empty(nbytes + 256, dtype=torch.uint8, device=gpu)
    buf = torch.full((B, Hq, 1, N), float("nan"), dtype=torch.float16, device=gpu)
    st = _native._I64x4(Hq * N, N, row_stride, 1)
    stream = torch.cuda.current_stream().cuda_stream
    if alone:
        rc = lib.fas_attention_scores(ctypes.byref(args), buf.data_ptr(), st, stream)
    else:
        rc = lib.fas_attention_with_scores(ctypes.byref(args), buf.data_ptr(), st,
                                           ws.data_ptr() + (-ws.data_ptr()) % 256, nbytes, stream)
    _native.check(lib, rc, "scores")
    torch.cuda.synchronize()
    heads = sorted({0, 1, Hq - 1})
    ref = naive.reference_forward(q, k, v, causal=True, want=("scores",), heads=heads)
    assert_scores_close(buf[:, heads], ref["scores"][:, heads])
