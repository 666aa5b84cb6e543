"""The prefill GEMMs at the edges of their tiles, K splits and value ranges,
against the oracle: block sums bit-exact, outputs within the
tolerance of an f32 sum in another order (tests/_metrics.py)."""
import numpy as np
import pytest

import oracle as O
from arm_ai_amd import synth as S
from tests.test_gpu_parity import check_matmul

pytestmark = pytest.mark.gpu

KQ = [S.TYPE_Q2_K, S.TYPE_Q3_K, S.TYPE_Q4_K, S.TYPE_Q5_K, S.TYPE_Q6_K]


# n: less than, exactly and past the 128- and 256-column tiles, rows not whole
# row blocks; k: one super-block, an odd count, enough for several splits;
# m: around the 32-, 64- and 128-row tiles
@pytest.mark.parametrize("t", KQ)
@pytest.mark.parametrize("n,k,m", [(5, 256, 9), (128, 768, 32), (129, 256, 33), (257, 1280, 65), (100, 4096, 64),
                                   (384, 2816, 129)])
def test_tile_edges(ctx, t, n, k, m):
    rng = np.random.default_rng(n * 7 + m)
    check_matmul(ctx, S.make_weight(t, n, k, rng=rng), S.make_activation(m, k, seed=m))


# the few-row forms: four and eight wavefronts over K, with and without a
# split, K from one super-block (idle wavefronts) to an odd count
@pytest.mark.parametrize("t", KQ)
@pytest.mark.parametrize("n,k,m", [(33, 256, 3), (70, 768, 5), (1000, 2304, 8), (2048, 5632, 17), (520, 3840, 40)])
def test_few_rows(ctx, t, n, k, m):
    rng = np.random.default_rng(n + 3 * m)
    check_matmul(ctx, S.make_weight(t, n, k, rng=rng), S.make_activation(m, k, seed=m + 1))


# many row and column tiles: the 128 x 256 form (outputs only: the dump has its own form)
@pytest.mark.parametrize("t", KQ)
def test_large_tiles(ctx, t):
    rng = np.random.default_rng(5)
    check_matmul(ctx, S.make_weight_unit(t, 9000, 768, rng=rng), S.make_activation(700, 768, seed=3), sums=False, cond=False)


# the largest quants, scales and mins under an activation of one sign: sums
# past 2^24, which the output's f32 chain rounds (by at most half an ulp of
# 2^26 per step, relative 2^-24) and the dump must hold exactly
@pytest.mark.parametrize("t", KQ)
def test_extreme_sums(ctx, t):
    W = S.make_weight(t, 40, 512, seed=1)
    if t == S.TYPE_Q4_K:
        blocks = S.pack_q4k(W.d, W.dmin, np.full_like(W.sc, 63), np.full_like(W.mn, 63), np.full_like(W.q, 15))
    elif t == S.TYPE_Q5_K:
        blocks = S.pack_q5k(W.d, W.dmin, np.full_like(W.sc, 63), np.full_like(W.mn, 63), np.full_like(W.q, 31))
    elif t == S.TYPE_Q6_K:
        blocks = S.pack_q6k(W.d, np.full_like(W.sc, -128), np.full_like(W.q, -32))
    elif t == S.TYPE_Q2_K:
        blocks = S.pack_q2k(W.d, W.dmin, np.full_like(W.sc, 15), np.full_like(W.mn, 15), np.full_like(W.q, 3))
    else:
        blocks = S.pack_q3k(W.d, np.full_like(W.sc, -32), np.full_like(W.q, -4))
    W.blocks = blocks
    x = np.full((20, 512), -1.0, np.float32)  # every quant -128
    x[1] = 1.0
    x[2, ::3] = 0.5
    check_matmul(ctx, W, x, cond=False)


# the Q8_0 GEMM and its few-row forms: rows of padded groups (k not a multiple
# of 256), idle wavefronts, row tiles of one row, more than 64 KiB of d in LDS
@pytest.mark.parametrize("t", [S.TYPE_Q8_0, S.TYPE_Q4_0, S.TYPE_Q5_0])
@pytest.mark.parametrize("n,k,m", [(33, 96, 4), (576, 576, 5), (1000, 2304, 8), (130, 1312, 33), (100, 14336, 7),
                                   (257, 1056, 65), (1536, 4096, 97), (520, 32, 200)])
def test_q8_rows(ctx, t, n, k, m):
    rng = np.random.default_rng(n + m)
    check_matmul(ctx, S.make_weight(t, n, k, rng=rng), S.make_activation(m, k, seed=m + 2))


def test_q8_large_tiles(ctx):
    rng = np.random.default_rng(9)
    check_matmul(ctx, S.make_weight(S.TYPE_Q8_0, 5000, 864, rng=rng), S.make_activation(500, 864, seed=1), sums=False, cond=False)
