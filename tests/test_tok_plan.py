"""The planner of the token-batched GEMV kernels (plan_tok), through the
measurement library and without a device, for a card of 256 CUs in 8 XCDs."""
import ctypes as C
import random

import pytest

from edgerunner_amd import _ffi

KINDS = {"q4_k": 0, "q8_0": 1, "q6_k": 2, "q8_rows": 3, "q8_pairs": 4}


def plan(kind, rows, K, T, mode=None, cu=256):
    """(row tiles, tokens, K slices, mode, workgroups, LDS, units per phase) or
    None where the one-token kernels keep the call; and the two estimates."""
    p, cost = (C.c_uint32 * 8)(), (C.c_float * 2)()
    lib = _ffi.load_probe()
    assert lib.er_hip_probe_tok_plan(KINDS[kind], rows, K, T, cu, mode.encode() if mode else None, p, cost) == 0
    return (tuple(p[1:]) if p[0] else None), tuple(cost)


def fullest_xcd(rows, T, split):
    """Workgroups of XCD 0: row block b runs on XCD b % 8, with all its token tiles."""
    rt, tt, kw = split[:3]
    blocks = -(-rows // (16 * rt * (8 // kw)))
    return -(-blocks // 8) * -(-T // tt)


@pytest.mark.parametrize("kind,rows,K,T", [("q8_0", 1289, 6400, 24), ("q4_k", 1291, 7680, 24)])
def test_a_round_is_the_fullest_xcds(kind, rows, K, T):
    """243 workgroups fit 256 CUs, but 33 of them are on the 32 CUs of XCD 0:
    two rounds, which is slower than the one-token kernels."""
    assert fullest_xcd(rows, T, (1, 8, 8)) == 33
    forced, cost = plan(kind, rows, K, T, "1:8:8")
    assert forced[:3] == (1, 8, 8)
    assert cost[0] > 1.5 * plan(kind, rows - 9 * 16, K, T, "1:8:8")[1][0]  # 9 row blocks less: one round
    assert plan(kind, rows, K, T)[0] is None


@pytest.mark.parametrize("kind,rows,K,T,taken", [
    ("q4_k", 289, 1024, 48, False), ("q4_k", 287, 1792, 48, False), ("q8_0", 625, 2816, 32, False),
    ("q8_0", 472, 11264, 32, False), ("q6_k", 703, 7680, 32, False),
    ("q4_k", 595, 512, 48, True), ("q6_k", 435, 8704, 77, True), ("q6_k", 428, 768, 77, True),
    ("q8_rows", 744, 15872, 77, True), ("q8_pairs", 660, 12288, 77, True)])
def test_short_matrices(kind, rows, K, T, taken):
    """Measured: the first five 18 to 26% slower on the token-batched kernels, the
    others 1.5 to 3 times faster."""
    assert (plan(kind, rows, K, T)[0] is not None) == taken


def test_taken_exactly_where_the_estimate_says():
    """The bound that turns small calls away before the search decides no call
    otherwise than the search does."""
    rng = random.Random(6)
    taken = 0
    for _ in range(4000):
        kind, T = rng.choice(list(KINDS)), int(2 ** rng.uniform(1, 7))
        rows, K = int(2 ** rng.uniform(6, 14)), 256 * int(2 ** rng.uniform(0, 6))
        best, one = plan(kind, rows, K, T, "1")[1]
        got = plan(kind, rows, K, T)[0]
        assert (got is not None) == (best < one), (kind, rows, K, T, best, one)
        taken += got is not None
    assert 500 < taken < 3500


def test_launches_are_the_kernels():
    """Whatever the shape: a built split, as many workgroups as its grid mapping
    needs, LDS within the CU's."""
    rng = random.Random(5)
    seen = 0
    for _ in range(4000):
        kind, T = rng.choice(list(KINDS)), rng.randint(2, 200)
        rows, K = int(2 ** rng.uniform(0, 17)) + rng.randint(0, 3), 256 * rng.randint(1, 64)
        got, _ = plan(kind, rows, K, T, rng.choice([None, "1"]))
        if got is None:
            continue
        seen += 1
        rt, tt, kw, mode, grid, lds, units = got
        assert (rt, tt) in {(1, 4), (4, 4), (1, 8), (4, 8), (1, 16), (2, 16)} and kw in (1, 2, 4, 8)
        assert grid == 8 * fullest_xcd(rows, T, got) and lds <= 163840 - 4096 and kw * units % 4 == 0
    assert seen > 1000
