"""Batches of 9 .. 64 tokens whose group scales are folded into the weights, two codes a multiplication (csrc/mmq_few.hip Planes): the ends of a byte's and a 16-bit lane's range."""
import numpy as np
import pytest

import oracle_py as oq
import np_twin as tw
from test_gpu_ops import BB, Q4_K, Q5_K, Q6_K, be  # noqa: F401
from test_gpu_few import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(256, 17, 9), (4096, 33, 16), (2048, 16, 17), (2304, 40, 33), (4096, 31, 48), (1024, 18, 49)])
def test_largest_codes_and_scales(be, t, K, N, T):  # noqa: F811
    """Codes, scales and activations at their largest, row by row of another sign or half: every integer of a super-block is exact, so the kernel that multiplies the sums by the
    scales has the same bits; the f32 order over super-blocks is all that is left to the oracle (2e-5 of the largest output, as for random weights)."""
    W = np.zeros(N * K // 256 * BB[t], np.uint8)
    blk = W.view(tw.DT[t]).reshape(N, K // 256)
    blk["d"] = np.float16(1e-2)
    for r in range(N):
        fill = (0xff, 0x0f, 0xf0, 0x77)[r % 4]                  # all codes at their largest; one half of them; half as large and one more
        if t == Q6_K:
            blk["ql"][r] = fill
            blk["qh"][r] = (0xff, 0x00, 0xff, 0xaa)[r % 4]
            blk["scales"][r] = (127, -128, -127, 127)[r % 3 if r % 4 else 1]
        else:
            blk["dmin"][r] = np.float16(1e-2)
            blk["scales"][r] = (0xff, 0x3f, 0xc0)[r % 3]
            blk["qs"][r] = fill
            if t == Q5_K:
                blk["qh"][r] = (0xff, 0x55, 0x00)[(r // 2) % 3]
    x = np.ones((T, K), np.float32) * (1.0 + np.arange(T, dtype=np.float32)[:, None])
    x[1::3] *= -1.0                                             # codes of -127, and of one sign after another
    x[2::3, ::2] *= -1.0
    y, other = both(be, lambda: be.mul_mat(t, W, N, K, x))
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
    assert np.array_equal(y, other)
