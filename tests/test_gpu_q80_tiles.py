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


SHAPES = [(16, [(256, 1, 3), (512, 40, 5), (768, 65, 16), (256, 1, 32), (256, 33, 33), (768, 40, 63), (2048, 130, 47), (5632, 70, 40), (28672, 40, 35)]),   # fewer steps than buffers, ragged rows and tokens
          (32, [(256, 2049, 257), (768, 1100, 513), (2048, 2000, 323), (256, 14000, 513)]),
          (64, [(768, 8193, 897), (256, 14000, 640), (256, 14070, 511), (512, 8200, 896), (2304, 8193, 895)])]                 # whole and ragged tiles; rows of two to eighteen steps through two buffers


@pytest.mark.parametrize("form,K,N,T", [(f, *c) for f, cs in SHAPES for c in cs])
def test_q80_tiles_bit_exact(be, form, K, N, T):  # noqa: F811
    """Integer block sums, three roundings a block, blocks in order: the oracle's bits, in tiles of 16, of 32 and of 2 x 2 times 32 a wave."""
    assert be.lib.mi355_debug_q80_plan(N, K, T) == form
    rng = np.random.default_rng(K + N + T)
    W = scaled(rng, rand_weights(rng, Q8_0, N * K), N, K)
    x = (rng.standard_normal((T, K)) * 10.0 ** rng.uniform(-6, 2, (T, 1))).astype(np.float32)
    x[T // 2] = 0
    assert np.array_equal(be.mul_mat(Q8_0, W, N, K, x), oq.mul_mat(Q8_0, W, N, K, x))


@pytest.mark.parametrize("form,K,N,T", [(16, 256, 40, 33), (32, 256, 2049, 300), (64, 256, 14070, 511)])
def test_q80_infinite_scales_stay_in_their_block(be, form, K, N, T):  # noqa: F811
    """A block whose scale is infinite or NaN says so in its own outputs only, with the oracle's infinities."""
    assert be.lib.mi355_debug_q80_plan(N, K, T) == form
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
