"""Token-batched GEMV kernels (two and more tokens): every row of every token
equals the one-token call of the same matrix bit for bit, over the addition
orders that M and K select (whole rows with one and several slots per lane,
K-sliced rows whose slices start at and inside a 256-weight unit), row and
token remainders, every compiled configuration and slice count, and x the
limbs cannot carry.  The one-token calls are themselves held to the oracle
(test_gpu_gemv.py, test_gpu_gemv_cuk.py, test_gpu_fused_q8.py)."""
import functools
import os

import numpy as np
import pytest

import edgerunner_amd.synth as synth
from edgerunner_amd import Context, FusedQ8Kernel, GEMVKernel
from oracle import ref
from conftest import rel_l2
from test_tok_plan import plan

pytestmark = pytest.mark.gpu

FMTS = ("q4_k", "q8_0", "q6_k")
NAME = {"q4_k": "Q4K", "q6_k": "Q6K", "q8_0": "Q8_0"}


def batched_and_single(ctx, fmt, W, x, M, K, T):
    """(batched [T, M], the T one-token calls [T, M])."""
    g = GEMVKernel(ctx)
    wb, xb, yb, y1 = ctx.upload(W), ctx.upload(x), ctx.alloc(4 * T * M), ctx.alloc(4 * T * M)
    try:
        yb.upload(np.full(T * M, np.float32(7e30)))
        getattr(g, f"encodeBatched{NAME[fmt]}Weights")(None, wb, xb, yb, T, M, K)
        for t in range(T):
            getattr(g, f"encode{NAME[fmt]}Weights")(None, wb, xb.view(4 * t * K, 4 * K), y1.view(4 * t * M, 4 * M), M, K)
        ctx.synchronize()
        return yb.download(np.float32).reshape(T, M), y1.download(np.float32).reshape(T, M)
    finally:
        for b in (wb, xb, yb, y1):
            b.free()


def forced(split):
    """A context whose calls of two and more tokens take these kernels: "1" with
    the planner's split, "rt:tt:kw" with this one where a shape allows it."""
    old = os.environ.get("ER_HIP_GEMV_TOK")
    os.environ["ER_HIP_GEMV_TOK"] = split
    try:
        return Context(0)
    finally:
        if old is None:
            os.environ.pop("ER_HIP_GEMV_TOK", None)
        else:
            os.environ["ER_HIP_GEMV_TOK"] = old


@pytest.fixture(scope="module")
def tok():
    c = forced("1")
    yield c
    c.close()


# K: lane trees of 64 .. 4 leaves, several slots per lane (2560 and 3072 with
# many rows), K-sliced rows (4096 Q4_K; 4352, 5120, 11008 start slices inside a
# unit; 14336 and 16384 need several LDS phases)
SHAPES = [(1, 256, 2), (17, 512, 3), (33, 1280, 9), (300, 1024, 5), (9000, 768, 4), (8192, 3072, 6), (10000, 2560, 3),
          (2100, 4096, 17), (515, 4352, 7), (260, 5120, 16), (130, 11008, 5), (100, 14336, 19), (40, 16384, 33)]


@pytest.mark.parametrize("M,K,T", SHAPES)
@pytest.mark.parametrize("fmt", FMTS)
def test_rows_equal_one_token_calls(tok, fmt, M, K, T):
    W = synth.weights(fmt, synth.seed(96, 1), M, K)
    x = synth.normal_f32(synth.seed(96, 2), T * K)
    x[K:2 * K] = -0.0  # a token of nothing: its rows keep the one-token call's zeros, sign and all
    got, one = batched_and_single(tok, fmt, W, x, M, K, T)
    assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
    rows = slice(0, min(M, 64))
    n = len(W) // M
    exp = np.stack([ref.gemv(fmt, W[:n * min(M, 64)], x[t * K:(t + 1) * K], min(M, 64), K) for t in (0, T - 1)])
    assert rel_l2(got[[0, T - 1]][:, rows], exp) < 1e-3


SPLITS = [(1, 4), (4, 4), (1, 8), (4, 8), (1, 16), (2, 16)]  # {row tiles, tokens}, with 1, 2, 4 or 8 slices of K
PLAIN, CHAINED, INSIDE = range(3)  # one slot per leaf, several, slices that start inside a unit


def reached(kind):
    """The (addition mode, row tiles, tokens, slices) that some shape can take:
    compiled, with enough leaves for the slices, and within the LDS."""
    few = {(PLAIN, 2, 16, 8)} if kind != "q4_k" else set()
    small = kind not in ("q4_k", "q8_0")  # chained slots of these: as INSIDE of Q8_0, without {4, 8}
    out = set()
    for rt, tt in SPLITS:
        for kw in (1, 2, 4, 8):
            out.add((PLAIN, rt, tt, kw))
            if kw == 1 or small:  # whole rows of Q4_K and Q8_0 chain on four lanes only
                out.add((CHAINED, rt, tt, kw))
            if kind != "q6_k":
                out.add((INSIDE, rt, tt, kw))
    if small:
        few |= {(CHAINED, 4, 8, kw) for kw in (1, 2, 4, 8)} | {(CHAINED, 2, 16, 8)}
    if kind not in ("q4_k", "q6_k"):
        few |= {(INSIDE, 4, 8, kw) for kw in (1, 2, 4, 8)} | {(INSIDE, 2, 16, 2), (INSIDE, 2, 16, 8)}
    return out - few


@functools.lru_cache(maxsize=None)
def split_case(fmt, M, K, T):
    return synth.weights(fmt, synth.seed(96, 3), M, K), synth.normal_f32(synth.seed(96, 4), T * K)


SPLIT_SHAPES = {"q4_k": [(70, 1024, 5), (9000, 512, 2), (9000, 256, 2), (50, 5120, 6), (45, 14336, 18)],
                "q8_0": [(70, 1024, 5), (9000, 512, 2), (9000, 256, 2), (50, 4352, 6), (45, 14336, 18)],
                "q6_k": [(40, 256, 5), (9000, 256, 2), (9000, 512, 5), (16500, 4352, 3), (45, 14336, 18), (8300, 12544, 2)]}


@pytest.mark.parametrize("rt,tt", SPLITS)
@pytest.mark.parametrize("fmt", FMTS)
def test_every_split(fmt, rt, tt):
    """Every compiled {row tiles, tokens} with every count of K slices that a
    shape can take, in each addition mode and over one and several phases.  A
    split that a shape does not take is left out: the call would run the
    one-token kernels."""
    ran = set()
    for kw in (1, 2, 4, 8):
        split = f"{rt}:{tt}:{kw}"
        c = forced(split)
        try:
            assert c.compute_units == 256
            for M, K, T in SPLIT_SHAPES[fmt]:
                p, _ = plan(fmt, M, K, T, split)
                if p is None:
                    continue
                assert p[:3] == (rt, tt, kw)
                got, one = batched_and_single(c, fmt, *split_case(fmt, M, K, T), M, K, T)
                assert np.array_equal(got, one), (kw, M, K, T, fmt)
                ran.add((p[3], rt, tt, kw))
        finally:
            c.close()
    assert ran == {r for r in reached(fmt) if r[1:3] == (rt, tt)}


@pytest.mark.parametrize("rt,tt", SPLITS)
def test_every_split_fused(rt, tt):
    """The same for the fused projections' rows and gate/up pairs."""
    ran = {"q8_rows": set(), "q8_pairs": set()}
    for kw in (1, 2, 4, 8):
        split = f"{rt}:{tt}:{kw}"
        c = forced(split)
        try:
            for q, kv, dim in ((40, 20, 256), (40, 20, 4352), (5000, 4500, 512), (4000, 4500, 256), (4000, 4500, 2304),
                               (4000, 4500, 6912), (45, 20, 14336)):
                taken = {k: plan(k, n, dim, 5, split)[0] for k, n in (("q8_rows", q + 2 * kv), ("q8_pairs", 2 * kv))}
                if not any(taken.values()):
                    continue
                x = synth.normal_f32(synth.seed(97, 7), 5 * dim).reshape(5, dim)
                check_fused(c, dim, q, kv, x, np.abs(synth.normal_f32(synth.seed(97, 8), dim)))
                for k, p in taken.items():
                    if p is not None:
                        ran[k].add((p[3], rt, tt, kw))
        finally:
            c.close()
    for k, r in ran.items():
        assert r == {w for w in reached(k) if w[1:3] == (rt, tt)}, k


@functools.lru_cache(maxsize=None)
def fused_weights(q, kv, dim):
    return [synth.q8_0(synth.seed(97, i), m, dim) for i, m in enumerate((q, kv, kv))]


def check_fused(ctx, dim, q, kv, x, nw):
    """RMSNorm + QKV (fp32 and fp16 V) and gate/up + SiLU of x [T, dim] against
    the one-token calls, bit for bit (any NaN equals any other); returns V in
    fp32 and the activations."""
    T = len(x)
    f = FusedQ8Kernel(ctx)
    W = fused_weights(q, kv, dim)
    b = [ctx.upload(a) for a in (*W, np.ascontiguousarray(x), nw)]
    sizes = (4 * q, 4 * kv, 2 * kv, 4 * kv, 4 * kv)  # q, k, v16, v32, act
    types = (np.float32, np.float32, np.float16, np.float32, np.float32)
    outs = [ctx.alloc(T * n) for n in sizes]
    one = [ctx.alloc(T * n) for n in sizes]

    def encode(xb, o, n):
        f.encodeFusedQKV(None, *b[:3], xb, o[0], o[1], o[2], b[4], q, kv, dim, n, 1e-5)
        f.encodeFusedQKVTurbo(None, *b[:3], xb, o[0], o[1], o[3], b[4], q, kv, dim, n, 1e-5)
        f.encodeFusedGateUpSilu(None, b[1], b[2], xb, o[4], b[4], kv, dim, n, 1e-5)
    try:
        encode(b[3], outs, T)
        for t in range(T):
            encode(b[3].view(4 * t * dim, 4 * dim), [o.view(t * n, n) for o, n in zip(one, sizes)], 1)
        ctx.synchronize()
        got = [o.download(ty).reshape(T, -1) for o, ty in zip(outs, types)]
        for g, w, ty in zip(got, one, types):
            assert np.array_equal(g, w.download(ty).reshape(T, -1), equal_nan=True)
        return got[3], got[4]
    finally:
        for buf in b + outs + one:
            buf.free()


@pytest.mark.parametrize("dim,q,kv,T", [(1024, 70, 30, 5), (2560, 5000, 1300, 3), (4096, 4096, 1024, 18),
                                        (5120, 300, 77, 6), (14336, 130, 40, 9), (14336, 2100, 40, 2)])
def test_fused_q8_rows_equal_one_token_calls(tok, dim, q, kv, T):
    """RMSNorm + QKV (fp32 and fp16 V) and gate/up + SiLU."""
    x = synth.normal_f32(synth.seed(97, 5), T * dim).reshape(T, dim)
    nw = (np.float32(0.5) + np.abs(synth.normal_f32(synth.seed(97, 6), dim))).astype(np.float32)
    check_fused(tok, dim, q, kv, x, nw)


@pytest.mark.parametrize("dim,q,kv", [(1024, 70, 30), (2560, 5000, 1300), (4096, 4096, 1024), (5120, 300, 77),
                                      (14336, 130, 40)])
def test_fused_x_the_limbs_cannot_carry(tok, dim, q, kv):
    """Tokens with NaN, with infinities, with outliers that send the call to its
    fp32 evaluation, and with a NaN and outliers, under RMSNorm: rows of every
    matrix and gate/up pairs equal the one-token calls bit for bit."""
    assert plan("q8_rows", q + 2 * kv, dim, 8, "1")[0] and plan("q8_pairs", 2 * kv, dim, 8, "1")[0]
    x = synth.normal_f32(synth.seed(97, 9), 8 * dim).reshape(8, dim)
    x[1, 5] = np.nan
    x[2, dim - 1], x[2, 70] = np.inf, -np.inf
    x[3, 64] = np.inf
    x[5, ::64] = 1e6
    x[6, ::64], x[6, dim - 2] = 1e6, np.nan
    nw = (np.float32(0.5) + np.abs(synth.normal_f32(synth.seed(97, 10), dim))).astype(np.float32)
    v, act = check_fused(tok, dim, q, kv, x, nw)
    for y in (v, act):
        assert np.isnan(y[[1, 6]]).all() and np.isfinite(y[[0, 4, 5, 7]]).all() and not np.isfinite(y[[2, 3]]).any()


@pytest.mark.parametrize("M,K", [(100, 1024), (2100, 4096), (60, 14336)])
@pytest.mark.parametrize("fmt", FMTS)
def test_x_the_limbs_cannot_carry(tok, fmt, M, K):
    """A token with NaN, one with infinities and one whose outliers send the
    launch to its fp32 evaluation: all equal the one-token calls bit for bit."""
    T = 6
    W = synth.weights(fmt, synth.seed(98, 1), M, K)
    x = synth.normal_f32(synth.seed(98, 2), T * K).reshape(T, K)
    x[1, 5] = np.nan
    x[2, K - 1], x[2, 70] = np.inf, -np.inf
    x[4, ::64] = 1e6
    got, one = batched_and_single(tok, fmt, W, x, M, K, T)
    assert np.array_equal(got, one, equal_nan=True)
    assert np.isnan(got[1]).all() and np.isfinite(got[[0, 3, 4, 5]]).all()


def _conditioning_x(K, f, half, T):
    """[T, K] whose tokens step across the rule that sends a call to its fp32
    evaluation, f (64 / 12) sum s_g^2 > 2^-24 sum rest_g, about 6e-8 of its right
    side apart: nearer than the order of its fp32 sums matters.  One outlier of
    1e5 in each 64-group gives every group the scale s_g = 2^-5; rest_g counts the
    squares outside the outlier's 16 (half: 8) values."""
    x = synth.normal_f32(synth.seed(99, 1), K).astype(np.float64)
    rest = x.reshape(-1, 64).copy()
    rest[:, :8 if half else 16] = 0.0
    lhs = f * (64.0 / 12.0) * (K / 64.0) * 2.0 ** -10
    a0 = np.sqrt(lhs / (float(np.float32(5.9604645e-08)) * (rest ** 2).sum()))
    out = np.empty((T, K), dtype=np.float32)
    for t in range(T):
        out[t] = (x * (a0 * (1.0 + (t - T / 2) * 2.0 ** -25))).astype(np.float32)
        out[t, ::64] = 1e5
    return out


# one-token kernels by how they convert x: 8 values a lane (K-sliced rows of
# 4096 and less, CU-resident ones of 2048 and less) or 16, in four waves, eight
# or one slice each
CONDITIONING = [("q4_k", 2100, 4096, True), ("q4_k", 16400, 1024, True), ("q6_k", 16400, 1024, True),
                ("q8_0", 5000, 4096, False), ("q4_k", 300, 1024, False), ("q6_k", 1000, 2048, False),
                ("q8_0", 300, 8192, False), ("q4_k", 260, 14336, False), ("q6_k", 300, 11008, False)]


@pytest.mark.parametrize("fmt,M,K,half", CONDITIONING)
def test_fp32_evaluation_decided_as_the_one_token_call(tok, fmt, M, K, half):
    """A second outlier beside a group's first, in the same 8 values, in the same
    16 only and in neither: whether the call falls back to fp32 depends on how
    its one-token kernel converts x, and batching must not change that; then
    tokens across the rule's threshold, where the order of its sums decides."""
    T = 6
    W = synth.weights(fmt, synth.seed(99, 2), M, K)
    x = synth.normal_f32(synth.seed(99, 3), T * K).reshape(T, K)
    x[1:, ::64] = 1e6
    for t, at in ((2, 7), (3, 8), (4, 15), (5, 16)):
        x[t, at::64] = 9e5
    got, one = batched_and_single(tok, fmt, W, x, M, K, T)
    assert np.array_equal(got, one)
    x = _conditioning_x(K, 1.0 if fmt == "q8_0" else 4.0, half, 64)
    got, one = batched_and_single(tok, fmt, W, x, M, K, 64)
    assert np.array_equal(got, one)


@pytest.mark.parametrize("dim", [1024, 4096, 5120])
def test_fused_fp32_evaluation_decided_as_the_one_token_call(tok, dim):
    """The same for the fused projections, whose rule sees x under RMSNorm
    (K-sliced rows: x times the norm weight, here powers of two)."""
    x = np.concatenate([synth.normal_f32(synth.seed(99, 4), 6 * dim).reshape(6, dim),
                        _conditioning_x(dim, 1.0, dim == 4096, 64)])
    x[1:6, ::64] = 1e6
    for t, at in ((2, 7), (3, 8), (4, 15), (5, 16)):
        x[t, at::64] = 9e5
    nw = np.exp2(np.floor(2.0 * np.abs(synth.normal_f32(synth.seed(99, 5), dim // 64)))).astype(np.float32)
    check_fused(tok, dim, 300, 120, x, np.repeat(nw, 64))
