"""The K-grouped prefill GEMM, forced on both of its token tiles
(ER_HIP_GEMM_VARIANT=6: 32 tokens, 7: 64) where it can go wrong: one token and
one past a tile, one row and one past a tile, K of one chunk (three of the four
groups have none), of five and seven chunks (a last step that not all groups
have) and of whole steps; then shapes that select it unforced, by their bits,
against the kernels that split K over workgroups.  Bars: 1e-5 against the float64 product
with the bf16-rounded weights, fp32 sums of at most 2048 products being within
2048 * 2^-24 = 1.2e-4 of the sum of magnitudes at the worst and about its
square root, 3e-6, as they come; two kernels are twice that apart."""
import numpy as np
import pytest

import edgerunner_amd.synth as synth
from oracle import restate_np as rn
from conftest import rel_l2
from test_gpu_gemm import DSCALE, bf16_round, bf16_to_f32
from test_gpu_gemm_variants import _gemm

pytestmark = pytest.mark.gpu


def _case(fmt, T, N, K):
    return (synth.weights(fmt, synth.seed(53, 0), N, K, **DSCALE[fmt]), synth.normal_bf16(synth.seed(53, 1), T * K))


@pytest.mark.parametrize("variant", ["6", "7"])
@pytest.mark.parametrize("fmt,T,N,K", [
    ("q8_0", 1, 1, 64), ("q8_0", 33, 65, 320), ("q8_0", 64, 63, 448), ("q8_0", 65, 130, 1024), ("q8_0", 31, 200, 2048),
    ("q4_k", 1, 1, 256), ("q4_k", 33, 65, 256), ("q4_k", 64, 63, 768), ("q4_k", 65, 130, 1024), ("q4_k", 31, 200, 2048)])
def test_forced(variant, fmt, T, N, K):
    c, gemm = _gemm(ER_HIP_GEMM_VARIANT=variant)
    try:
        W, X = _case(fmt, T, N, K)
        Y = gemm.execute(fmt, W, X, T, N, K)
        again = gemm.execute(fmt, W, X, T, N, K)
    finally:
        c.close()
    exact = bf16_to_f32(X).reshape(T, K).astype(np.float64) @ bf16_round(rn.weights_f32(fmt, W, N, K)).astype(np.float64).T
    assert rel_l2(Y, exact) < 1e-5
    assert np.array_equal(Y, again)


@pytest.mark.parametrize("fmt", ["q4_k", "q8_0"])
@pytest.mark.parametrize("T,N,K,tile", [(16, 1024, 1024, 32), (100, 2048, 1024, 32), (128, 1032, 512, 32),
                                        (257, 3072, 1024, 64), (60, 14336, 256, 64)])
def test_selected_against_the_split(fmt, T, N, K, tile):
    assert T * N % 4 == 0  # else the forced split would not split
    W, X = _case(fmt, T, N, K)
    out = []
    for env in ({}, {"ER_HIP_GEMM_VARIANT": "6" if tile == 32 else "7"}, {"ER_HIP_GEMM_TILE": "64:4"}):
        c, gemm = _gemm(**env)
        try:
            out.append(gemm.execute(fmt, W, X, T, N, K))
        finally:
            c.close()
    # the sums of the K-grouped kernel in its own order: it is the one that ran
    assert np.array_equal(out[0], out[1]) and not np.array_equal(out[0], out[2])
    assert rel_l2(out[0], out[2]) < 2e-5
