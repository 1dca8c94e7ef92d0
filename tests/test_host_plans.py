"""The launches that the C ABI's host code plans, without a GPU.

fas_api.cpp is compiled with stand-ins for the kernel launchers
(tests/plans/launch_log.cpp) that log each launch's mode, row blocks and
splits.  Requests carry fake pointers that nothing dereferences.  Every call
takes the workspace that fas_workspace_bytes asks for, as the launchers do.
"""
from __future__ import annotations

import ctypes
import os
import random
import subprocess

import pytest

from flash_attn_with_score_amd import _native
from flash_attn_with_score_amd.csrc import build as fas_build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PTR = 0x1000000  # 256-byte aligned
PLAIN, SCORES, ROWSUM, FEW = 0, 1, 2, 5  # FwdMode


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("plans")
    flags = ["-O1", "-std=c++17", "-fPIC", f"--offload-arch={fas_build.ARCH}",
             f"-I{os.path.join(ROOT, 'include')}", f"-I{fas_build.CSRC}"]
    objs = []
    for src in (fas_build.CSRC / "fas_api.cpp", os.path.join(ROOT, "tests/plans/launch_log.cpp")):
        objs.append(str(tmp / (os.path.basename(src) + ".o")))
        subprocess.run([fas_build.hipcc(), "-x", "hip", *flags, "-c", str(src), "-o", objs[-1]],
                       check=True, capture_output=True, text=True)
    so = str(tmp / "plans.so")
    subprocess.run([fas_build.hipcc(), "-shared", "-fPIC", f"--offload-arch={fas_build.ARCH}",
                    "-Wl,-Bsymbolic", *objs, "-o", so], check=True, capture_output=True, text=True)
    lib = ctypes.CDLL(so)
    for name, (restype, argtypes) in _native._SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = restype, argtypes
    lib.plan_log_take.restype = ctypes.c_char_p
    return lib


def make_args(B, Hq, Hk, M, N, D, causal=1, dropout=0.0, dtype=1):
    a = _native.AttnArgs()
    a.dtype, a.causal, a.sm_scale = dtype, causal, D ** -0.5
    a.batch, a.heads_q, a.heads_k, a.seqlen_q, a.seqlen_k, a.head_dim = B, Hq, Hk, M, N, D
    a.q = a.k = a.v = a.out = PTR
    for name, H, L in (("q_stride", Hq, M), ("k_stride", Hk, N), ("v_stride", Hk, N),
                       ("out_stride", Hq, M)):
        setattr(a, name, _native._I64x4(H * L * D, L * D, D, 1))
    a.dropout_p = dropout
    return a


def take(lib):
    """The logged launches: [(name, {field: value})]."""
    out = []
    for line in lib.plan_log_take().decode().splitlines():
        name, *fields = line.split()
        out.append((name, {k: int(v) for k, v in (f.split("=") for f in fields)}))
    return out


def launches(lib, entry, a, split=0):
    """Sends one request with the workspace it asks for; returns its launches."""
    B, H, Hk, M, N = a.batch, a.heads_q, a.heads_k, a.seqlen_q, a.seqlen_k
    q4, k4 = a.q_stride, a.k_stride
    rows, keys = _native._I64x3(H * M, M, 1), _native._I64x3(Hk * N, N, 1)
    s4 = _native._I64x4(H * M * N, M * N, N, 1)
    variant = getattr(_native, "VARIANT_" + entry.upper().replace("_NOALLOC", ""))
    nbytes = lib.fas_workspace_bytes(variant, ctypes.byref(a), split)
    ws = (PTR, nbytes, None)
    ref = ctypes.byref(a)
    take(lib)
    if entry == "scores":
        rc = lib.fas_attention_with_scores(ref, PTR, s4, *ws)
    elif entry == "row_sum":
        rc = lib.fas_attention_with_row_sum(ref, PTR, rows, *ws)
    elif entry == "softmax_col_sum":
        rc = lib.fas_attention_with_softmax_col_sum(ref, PTR, keys, *ws)
    elif entry == "softmax_col_sum_noalloc":
        rc = lib.fas_attention_with_softmax_col_sum_noalloc(ref, PTR, keys, None)
    elif entry == "cross_softmax_sum":
        rc = lib.fas_attention_cross_token_softmax_sum(ref, split, PTR,
                                                       _native._I64x3(Hk * split, split, 1), *ws)
    elif entry == "attention_forward":
        rc = lib.fas_attention_forward(ref, PTR, rows, *ws)
    elif entry == "attention_backward":
        rc = lib.fas_attention_backward(ref, PTR, q4, PTR, rows, PTR, q4, PTR, k4, PTR, k4, *ws)
    else:
        raise ValueError(entry)
    assert rc == 0, _native.last_error(lib)
    return take(lib)


# (B, Hq, Hk, M, N, D): many query heads per KV head over few rows, with
# unaligned and whole score rows.
@pytest.mark.parametrize("shape", [(64, 32, 1, 2, 4100, 64), (32, 16, 1, 3, 8192, 128),
                                   (24, 64, 1, 8, 12001, 32), (40, 40, 2, 5, 5001, 16)])
def test_scores_pack_at_most_eight_heads(lib, shape):
    """The resident-Q scores kernel packs up to eight query heads of a KV head
    (a power of two); more of them run as several groups and are not refused."""
    a = make_args(*shape)
    B, H, Hk, M, N, D = shape
    rc = lib.fas_attention_scores(ctypes.byref(a), PTR, _native._I64x4(H * M * N, M * N, N, 1), None)
    assert rc == 0, _native.last_error(lib)
    sc = [f for name, f in take(lib) + launches(lib, "scores", a) if name == "scores"]
    assert sc and all(f["pshift"] <= 3 and (H // Hk) % (1 << f["pshift"]) == 0 for f in sc)


# (B, Hq, Hk, M, N, D) with at most 64 row blocks of 256
@pytest.mark.parametrize("shape", [(1, 1, 1, 4096, 4096, 64), (1, 4, 4, 64, 1024, 64),
                                   (1, 16, 16, 1024, 4096, 128), (1, 8, 2, 2048, 2048, 32),
                                   (2, 12, 12, 48, 1600, 128)])
def test_scores_with_dropout_split_keys(lib, shape):
    """Few row blocks with dropout: a key-split forward and the scores-only
    kernel, not the fused writer's 256-row blocks (split / fused, us: 57 / 290
    at B1 H1 S4096 D64)."""
    plan = launches(lib, "scores", make_args(*shape, dropout=0.1))
    assert [(n, f.get("mode", PLAIN)) for n, f in plan] == [("fwd", PLAIN), ("scores", PLAIN)]
    many = launches(lib, "scores", make_args(4, 32, 32, 1024, 1024, 64, dropout=0.1))
    assert [f["mode"] for _, f in many] == [SCORES]


# (B, Hq, Hk, M, N, D), the forward's mode, rows per block
SCORES_PLANS = [
    ((1, 1, 1, 4096, 4096, 128), PLAIN, None),   # 16 row blocks over 4096 keys: split
    ((1, 4, 4, 512, 3000, 128), PLAIN, None),    # 8 over 3000
    ((1, 4, 4, 2048, 2048, 128), SCORES, 64),    # 32 over 2048: fused
    ((1, 12, 12, 1024, 4096, 64), SCORES, 64),   # 48 over 4096
    ((1, 4, 4, 4096, 16384, 128), PLAIN, None),  # 64 over 16384
    ((2, 12, 12, 48, 1300, 128), PLAIN, None),   # up to 128 rows below 2048 keys
    ((2, 12, 12, 48, 1600, 64), PLAIN, None),
    ((2, 12, 12, 48, 1600, 32), SCORES, 64),
    ((2, 12, 12, 48, 1900, 32), PLAIN, None),
    ((2, 12, 12, 160, 1900, 128), SCORES, 64),
    ((1, 4, 4, 1, 1000, 128), FEW, None),        # few rows below 2048 keys
    ((1, 4, 4, 1, 1024, 64), SCORES, 64),
    ((1, 8, 1, 4, 1300, 16), FEW, None),
    ((16, 12, 12, 2, 2000, 128), SCORES, 64),    # 192 row blocks
    ((2, 12, 12, 48, 1024, 128), SCORES, 64),
    ((64, 32, 1, 1, 1000, 64), FEW, None),       # 2048 heads: the fused writer needs 8 rounds
    ((64, 32, 1, 1, 960, 64), SCORES, 256),
    ((2, 12, 12, 700, 2048, 32), SCORES, 64),    # D = 32: 264 blocks of 64
    ((2, 12, 12, 700, 2048, 128), SCORES, 128),
    ((1, 28, 28, 1024, 4096, 32), SCORES, 128),  # 448 blocks of 64
    ((4, 8, 8, 2048, 4096, 128), SCORES, 256),   # two full rounds of 128, the mask cuts little
    ((1, 32, 8, 2048, 8192, 32), SCORES, 128),   # D = 32: longer rows than that
    ((1, 32, 8, 2048, 8192, 64), SCORES, 256),
    ((1, 36, 36, 1024, 2048, 128), SCORES, 128),
    ((1, 32, 32, 2048, 3072, 128), SCORES, 128),
    ((1, 16, 16, 4096, 4096, 128), SCORES, 128),
]


@pytest.mark.parametrize("shape,mode,bm", SCORES_PLANS)
def test_scores_route_and_row_blocks(lib, shape, mode, bm):
    """Key split or fused writer, and the writer's row blocks, on both sides of
    each measured line."""
    name, f = launches(lib, "scores", make_args(*shape))[0]
    assert name == "fwd" and f["mode"] == mode
    if mode == SCORES:
        assert f["bm"] == bm


# (B, Hq, Hk, S, D, causal), pieces
PIECES = [
    ((1, 64, 1, 1024, 128, 1), 49),  # up to one per query head
    ((1, 32, 1, 2048, 64, 1), 32),
    ((1, 16, 1, 2048, 128, 0), 16),
    ((1, 8, 4, 2048, 64, 1), 8),     # more than the group's heads
    ((1, 4, 4, 1024, 64, 1), 4),     # one head of 16 row tiles: at least 4 a piece
    ((4, 32, 32, 4096, 64, 0), 1),   # the chip is full
]


@pytest.mark.parametrize("shape,pieces", PIECES)
def test_dkdv_pieces(lib, shape, pieces):
    """Workgroups per key block and KV head of the dK/dV kernel, and a
    workspace that holds exactly their partials."""
    B, Hq, Hk, S, D, causal = shape
    a = make_args(B, Hq, Hk, S, S, D, causal)
    (_, f), = launches(lib, "attention_backward", a)
    assert f["pieces"] == pieces
    r256 = lambda x: (x + 255) // 256 * 256  # noqa: E731
    rows = 2 * r256(B * Hq * ((S + 127) // 128 * 128) * 4)
    parts = r256(B * Hk * pieces * S * 2 * D * 4) if pieces > 1 else 0
    assert lib.fas_workspace_bytes(_native.VARIANT_ATTENTION_BACKWARD, ctypes.byref(a), 1) == \
        rows + parts


# entry, (B, Hq, Hk, M, N, D, causal, dropout), rows per block, splits
FWD_PLANS = [
    ("row_sum", (1, 4, 4, 1, 8192, 128, 1, 0.0), 256, 32),
    ("row_sum", (1, 8, 1, 4, 32768, 32, 1, 0.0), 256, 64),     # not 256: the merge is serial
    ("row_sum", (8, 32, 8, 1, 32768, 16, 1, 0.0), 256, 8),     # D <= 32: 512 workgroups at once
    ("row_sum", (8, 32, 8, 1, 32768, 64, 1, 0.0), 256, 4),
    ("row_sum", (4, 16, 16, 1000, 6000, 16, 0, 0.0), 128, 1),  # 512 blocks, one round
    ("row_sum", (4, 16, 16, 1000, 6000, 128, 0, 0.0), 256, 1),
    ("row_sum", (1, 4, 4, 128, 1024, 128, 1, 0.0), 256, 2),    # one wave per SIMD
    ("row_sum", (1, 4, 4, 512, 1024, 128, 1, 0.0), 128, 1),
    ("row_sum", (1, 32, 32, 128, 1024, 64, 1, 0.1), 256, 2),   # dropout: two CUs, not two waves
    ("row_sum", (1, 32, 32, 128, 1024, 64, 1, 0.0), 128, 1),
    ("softmax_col_sum", (1, 12, 12, 40, 1000, 32, 1, 0.1), 256, 2),
    ("scores", (1, 4, 4, 64, 1024, 64, 1, 0.1), 256, 2),
    ("attention_forward", (1, 4, 4, 127, 1090, 64, 1, 0.1), 256, 2),
    ("attention_forward", (1, 4, 4, 127, 1000, 64, 1, 0.0), 128, 1),
    ("attention_forward", (1, 32, 8, 127, 1090, 64, 1, 0.0), 128, 1),
    ("attention_forward", (1, 4, 4, 1531, 1531, 64, 1, 0.1), 256, 3),
    ("attention_forward", (1, 16, 16, 1531, 1531, 16, 1, 0.1), 256, 3),  # 288 workgroups
    ("row_sum", (1, 1, 1, 4096, 16384, 64, 1, 0.1), 256, 16),  # 18 would have 252 of 288
    ("row_sum", (1, 32, 1, 1, 4096, 16, 1, 0.0), 256, 16),     # whole eights of splits
]


@pytest.mark.parametrize("entry,shape,bm,nsplit", FWD_PLANS)
def test_forward_plan(lib, entry, shape, bm, nsplit):
    """Rows per workgroup and key splits of the forward around its measured lines."""
    B, Hq, Hk, M, N, D, causal, dropout = shape
    _, f = launches(lib, entry, make_args(B, Hq, Hk, M, N, D, causal, dropout))[0]
    assert (f["bm"], f["nsplit"]) == (bm, nsplit)


@pytest.mark.parametrize("seed", range(4))
def test_column_pass_split(lib, seed):
    """The column pass's workgroups per unit against the rule restated in
    test_host, over shapes that leave CUs idle, fill them and take rounds."""
    from tests.test_host import _col_plan

    rng = random.Random(seed)
    shapes = [(1, 28, 4, 4096, 4096, 0), (2, 28, 4, 1531, 1531, 0), (1, 32, 32, 3000, 3000, 2250),
              (1, 8, 2, 1024, 1024, 0), (1, 2, 2, 1300, 1300, 0), (1, 16, 1, 3000, 3000, 0)]
    for _ in range(60):
        Hk, G = rng.choice([1, 2, 4, 8, 12, 32]), rng.choice([1, 2, 3, 4, 7, 8])
        M, N = rng.randint(40, 5000), rng.randint(40, 5000)
        shapes.append((rng.choice([1, 2, 4]), Hk * G, Hk, M, N, rng.choice([0, 0, rng.randint(1, N)])))
    for B, Hq, Hk, M, N, split in shapes:
        causal = rng.choice([0, 1])
        a = make_args(B, Hq, Hk, M, N, 64, causal)
        plan = launches(lib, "cross_softmax_sum" if split else "softmax_col_sum", a, split)
        if plan[-1][0] != "colsm":  # few rows: their scores are kept
            assert not split and Hq // Hk * M <= 32
            continue
        want = _col_plan(B, Hq, Hk, split or N, False, M, N, causal, split)[0]
        assert plan[-1][1]["nsplit"] == want, (B, Hq, Hk, M, N, causal, split)
        assert plan[-1][1]["fold"] == Hq // Hk


# (B, Hq, Hk, M, N), whether the scores are kept, least splits
NOALLOC = [((8, 32, 8, 1, 8192), 1, 4), ((8, 32, 8, 1, 32768), 1, 4), ((8, 32, 8, 1, 60000), 0, 4),
           ((1, 32, 8, 1, 400000), 1, 16), ((1, 32, 8, 1, 500000), 0, 32),
           ((1, 8, 8, 4, 500000), 1, 16)]


@pytest.mark.parametrize("shape,kept,nsplit", NOALLOC)
def test_kept_scores_leave_room_for_the_split(lib, shape, kept, nsplit):
    """In 64 MiB of scratch, few rows' scores are kept only where the key split's
    partials fit beside them: near the limit the forward keeps its splits."""
    plan = launches(lib, "softmax_col_sum_noalloc", make_args(*shape, 128))
    (name, f), second = plan
    assert name == "fwd" and f["kept"] == kept and f["mode"] == (FEW if kept else PLAIN)
    assert second[0] == ("few_cols" if kept else "colsm")
    assert f["nsplit"] >= nsplit


def test_kept_scores_stay_below_4_gib(lib):
    """Kept scores of 4 GiB and less; past that the column pass reads K."""
    below, past = ((64, 32, 8, 1, n, 128) for n in (524288, 524352))
    for shape, kept in ((below, 1), (past, 0)):
        a = make_args(*shape)
        assert launches(lib, "softmax_col_sum", a)[0][1]["kept"] == kept
    nbytes = lib.fas_workspace_bytes(_native.VARIANT_SOFTMAX_COL_SUM, ctypes.byref(a), 0)
    assert nbytes < 1 << 30


@pytest.mark.parametrize("seed", range(3))
def test_planned_launches_are_taken(lib, seed):
    """Random requests: every planned launch is one that its launcher takes (the
    row blocks, packings and splits that have instances), also from workspaces
    for one head at a time and with unaligned score rows."""
    rng = random.Random(100 + seed)
    for _ in range(400):
        Hk, G = rng.choice([1, 1, 2, 3, 8, 32]), rng.choice([1, 1, 2, 3, 4, 7, 8, 16, 32, 64])
        M = rng.choice([1, 2, 5, 32, 33, rng.randint(1, 300), rng.randint(1, 5000)])
        N = rng.choice([1, 63, 64, rng.randint(1, 1200), rng.randint(1, 40000)])
        B, D = rng.choice([1, 1, 2, 16, 64]), rng.choice([16, 32, 64, 128])
        causal, dropout = rng.choice([0, 1]), rng.choice([0.0, 0.0, 0.2])
        entry = rng.choice(["scores", "scores", "row_sum", "softmax_col_sum", "attention_forward",
                            "attention_backward", "cross_softmax_sum"])
        split = rng.randint(1, N) if entry == "cross_softmax_sum" else 0
        a = make_args(B, Hk * G, Hk, M, N, D, causal, dropout)
        case = (entry, B, Hk * G, Hk, M, N, D, causal, dropout, split)
        for name, f in launches(lib, entry, a, split):
            if name == "fwd":
                assert f["nsplit"] >= 1 and f["nrb"] == -(-M * f["pack"] // f["bm"]), case
                assert f["pack"] == 1 or not dropout, case
                if f["nsplit"] > 1:
                    assert f["bm"] == 256 and f["mode"] != SCORES, case
                    assert (f["nsplit"] - 1) * f["tps"] < -(-N // 64) <= f["nsplit"] * f["tps"], case
                if f["mode"] == SCORES:
                    assert f["bm"] == 256 or (f["bm"] in (64, 128) and f["pack"] == 1
                                              and not dropout), case
                elif f["bm"] != 256:
                    assert f["bm"] == 128 and f["mode"] in (PLAIN, ROWSUM, 4), case
                if f["mode"] == FEW:
                    assert f["pack"] == G and G * M <= 32 and not dropout and f["bm"] == 256, case
            elif name == "scores" and f["ngrp"] > 0:
                assert f["ngrp"] <= f["nkb"] and f["pshift"] <= 3, case
                assert G % (1 << f["pshift"]) == 0 and M << f["pshift"] <= 512, case
            elif name == "colsm":
                assert 1 <= f["nsplit"] <= 8 * G, case
            elif name == "bwd":
                assert 1 <= f["pieces"] <= max(8, G), case
