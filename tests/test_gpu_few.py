"""Batches of 3 .. 64 tokens against K-quant weights (csrc/mmq_few.hip): the contraction whose workgroups walk 16-row tiles with the quantiser's operand blocks."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import Q4_K, Q5_K, Q6_K, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(4096, 40, 4), (256, 8210, 3),       # a few rows; one super-block, more row tiles than workgroups, a ragged last one
                                   (4096, 4200, 16), (2048, 8193, 17),  # a full token tile and one token more; two super-blocks per wave and one, several tiles each
                                   (3584, 4130, 32), (11008, 50, 33),   # super-blocks that do not divide by the waves, up to two and more than two per wave
                                   (1024, 4113, 48), (4096, 17, 49), (5632, 4112, 64)])
def test_few_tokens(be, t, K, N, T):  # noqa: F811
    """Against the oracle: the integer of every super-block is exact and the fold the CPU's, so only the f32 order over super-blocks differs (eight partial sums of
    K / 256 / 8 terms, then eight terms: each f32 rounding is half an ulp, 2e-5 of the largest output as for the other contractions)."""
    rng = np.random.default_rng(5 * K + N + T + t)
    W = rand_weights(rng, t, N * K)
    x = (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)
    y = be.mul_mat(t, W, N, K, x)
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
