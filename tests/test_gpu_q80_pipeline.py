"""Prompt batches against Q8_0 weights (csrc/mmq_q80.hip): rows of one, eight and nine steps in tiles of 16, of two, four and eighteen in tiles of 32."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import Q8_0, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,T", [(256, 129, 32), (2048, 40, 33), (2304, 130, 65),       # tiles of 16, ragged rows and tokens
                                   (512, 8200, 250), (256, 16390, 250), (2304, 16384, 129)])  # a tile of 32 a wave
def test_q80_groups_bit_exact(be, K, N, T):  # noqa: F811
    """Integer block sums, three roundings a block, blocks in order: the oracle's bits."""
    rng = np.random.default_rng(K + N + T)
    W = rand_weights(rng, Q8_0, N * K)
    x = (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)
    y = be.mul_mat(Q8_0, W, N, K, x)
    assert np.array_equal(y, oq.mul_mat(Q8_0, W, N, K, x))
