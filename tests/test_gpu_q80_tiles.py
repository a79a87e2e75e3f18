"""Prompt batches against Q8_0 rows (csrc/mmq_q80.hip): tiles through LDS, the scales' products from the matrix unit."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import Q8_0, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


def scaled(rng, W, N, K):
    """Block scales of every kind that a file can hold: subnormal, zero, negative, the largest that keep sums finite."""
    d = W.reshape(N * K // 32, 34)[:, :2].view(np.float16)
    kind = rng.integers(0, 6, d.shape[0])
    d[kind == 0, 0] = np.float16(2.0 ** -24) * rng.integers(1, 1024, (kind == 0).sum()).astype(np.float16)
    d[kind == 1, 0] = 0
    d[kind == 2, 0] *= -1
    d[kind == 3, 0] = 60000
    return W


@pytest.mark.parametrize("K,N,T", [(256, 1, 3), (512, 40, 5), (768, 65, 16), (256, 1, 32), (256, 33, 33), (768, 40, 63), (2048, 130, 47), (5632, 70, 40), (28672, 40, 35),   # 16 x 16 tiles: fewer steps than buffers, ragged rows and tokens
                                   (256, 2049, 257), (768, 1100, 513), (2048, 2000, 323),                           # one 32 x 32 tile a wave
                                   (256, 14000, 513), (768, 8193, 897)])                                            # four
def test_q80_tiles_bit_exact(be, K, N, T):  # noqa: F811
    """Integer block sums, three roundings a block, blocks in order: the oracle's bits, whichever kernel takes the shape."""
    rng = np.random.default_rng(K + N + T)
    W = scaled(rng, rand_weights(rng, Q8_0, N * K), N, K)
    x = (rng.standard_normal((T, K)) * 10.0 ** rng.uniform(-6, 2, (T, 1))).astype(np.float32)
    x[T // 2] = 0
    assert np.array_equal(be.mul_mat(Q8_0, W, N, K, x), oq.mul_mat(Q8_0, W, N, K, x))


@pytest.mark.parametrize("K,N,T", [(256, 40, 33), (256, 2049, 300), (256, 14000, 513)])
def test_q80_infinite_scales_stay_in_their_block(be, K, N, T):  # noqa: F811
    """A block whose scale is infinite or NaN says so in its own outputs only, with the oracle's infinities."""
    rng = np.random.default_rng(K + N)
    W = rand_weights(rng, Q8_0, N * K)
    d = W.reshape(N, K // 32, 34)[:, :, :2].view(np.float16)
    d[3, 1] = np.inf
    d[7, 2] = -np.inf
    d[N - 1, 0] = np.nan
    x = rng.standard_normal((T, K)).astype(np.float32)
    with np.errstate(all="ignore"):
        want = oq.mul_mat(Q8_0, W, N, K, x)
    got = be.mul_mat(Q8_0, W, N, K, x)
    assert np.array_equal(got, want, equal_nan=True)
