"""Which contraction a batch takes (host logic: no GPU): the sides on which measured launches were the faster ones."""
import ctypes as C

import pytest

Q4_K, Q5_K, Q6_K = 12, 13, 14
MATVEC, FEW, KSPLIT, PLANES = 0, 1, 2, 3


@pytest.fixture(scope="module")
def plan(pkg):
    lib = pkg.load_library()
    return lambda *a: int(lib.mi355_debug_batch_plan(*a))


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("n", [129, 145, 200, 256])
def test_from_129_tokens_by_time(plan, t, n):
    """A tensor whose 128 x 256 tiles leave most of the chip idle stays with the K-split kernel; one that fills it (alone, K split, or as a SwiGLU pair) does not."""
    for rows, cols in [(2048, 2048), (2560, 2048), (2048, 5632), (1536, 8960), (2560, 2560), (1024, 8192)]:
        for sum_free in (0, 1):
            assert plan(t, rows, cols, n, 0, sum_free) == KSPLIT, (rows, cols)
    for rows, cols in [(6144, 4096), (4096, 14336), (4096, 11008), (8192, 8192), (8192, 28672), (8192, 1024), (32000, 4096)]:
        for sum_free in (0, 1):
            assert plan(t, rows, cols, n, 0, sum_free) == PLANES, (rows, cols)
    for rows, cols in [(5632, 2048), (8960, 1536), (8192, 3072), (14336, 4096), (18944, 3584)]:
        assert plan(t, rows, cols, n, 1, 0) == PLANES, (rows, cols)
    assert plan(t, 1024, 2048, n, 1, 0) == KSPLIT


def test_around_the_ranges_ends(plan):
    """One row is a mat-vec, and two of fewer than 1280 columns; from 257 tokens on the K-split kernel is out, whatever the shape."""
    assert [plan(Q4_K, 2048, 2048, n, 0, 0) for n in (1, 2, 3, 128, 129, 256, 257)] == [MATVEC, FEW, FEW, KSPLIT, KSPLIT, KSPLIT, PLANES]
    for t in (Q4_K, Q5_K, Q6_K):
        assert [plan(t, r, c, 2, p, 0) for r, c, p in [(4096, 1280, 0), (128256, 4096, 0), (14336, 4096, 1), (4096, 1024, 0), (2816, 1024, 1)]] == [FEW, FEW, FEW, MATVEC, MATVEC]
    assert plan(10, 4096, 4096, 2, 0, 0) == MATVEC            # (Q2_K has no contraction of few tokens)
    assert [plan(Q4_K, 8192, 4096, n, 0, 0) for n in (65, 128, 129)] == [PLANES] * 3
    assert plan(Q4_K, 2048, 2000, 64, 0, 0) == MATVEC


def test_to_64_tokens_by_shape(plan):
    """mmq_few.hip to 16 tokens; beyond, where its row tiles fill their rounds of CUs (Q6_K: one round), and from 49 on for gate | up and long rows of few tensors."""
    assert all(plan(t, n, 4096, T, 0, 0) == FEW for t in (Q4_K, Q5_K, Q6_K) for n in (512, 5120, 128256) for T in (3, 16))
    assert [plan(Q4_K, n, 5120, T, 0, 0) for n in (4096, 5120, 6144) for T in (17, 48)] == [FEW, FEW, KSPLIT, KSPLIT, FEW, FEW]
    assert [plan(Q6_K, n, 4096, T, 0, 0) for n in (4096, 6144, 128256) for T in (17, 48)] == [FEW, FEW, KSPLIT, KSPLIT, KSPLIT, KSPLIT]
    for T in (49, 64):
        assert [plan(t, 4096, 14336, T, 0, 0) for t in (Q4_K, Q5_K, Q6_K)] == [FEW, FEW, KSPLIT]
        assert [plan(Q4_K, r, c, T, 0, 0) for r, c in [(4096, 4096), (8192, 28672), (152064, 3584)]] == [KSPLIT] * 3
        assert [plan(t, 14336, 4096, T, 1, 0) for t in (Q4_K, Q5_K, Q6_K)] == [FEW, FEW, KSPLIT]


@pytest.mark.parametrize("n", [65, 96, 128])
def test_from_65_tokens_by_time(plan, n):
    """The 128 x 256 tiles take what fills the chip, K split, from 65 tokens on: at these sizes measured at half to nine tenths of the K-split kernel's time."""
    for t in (Q4_K, Q5_K, Q6_K):
        for rows, cols in [(2048, 2048), (2560, 2048), (2048, 5632), (4096, 4096), (3072, 3072)]:
            assert [plan(t, rows, cols, n, 0, s) for s in (0, 1)] == [KSPLIT] * 2, (rows, cols)
        for rows, cols in [(6144, 4096), (12288, 4096), (5120, 5120), (8192, 8192)]:
            assert [plan(t, rows, cols, n, 0, s) for s in (0, 1)] == [PLANES] * 2, (rows, cols)
        for rows, cols in [(8192, 3072), (14336, 4096), (28672, 8192)]:
            assert plan(t, rows, cols, n, 1, 0) == PLANES, (rows, cols)
        assert plan(t, 1024, 2048, n, 1, 0) == KSPLIT


@pytest.mark.parametrize("n", [65, 80, 96, 112, 128])
def test_from_65_tokens_by_the_bytes_of_a_type(plan, n):
    """Q6_K reaches the tiles as two bytes a weight: gate | up of 5632 x 2048, and the long rows of few tensors, stay with the K-split kernel where a Q4_K tensor does not."""
    assert plan(Q6_K, 5632, 2048, n, 1, 0) == KSPLIT
    for rows, cols in [(2048, 5632), (1536, 8960), (3072, 8192), (4096, 11008), (4096, 14336), (3584, 18944)]:
        assert plan(Q6_K, rows, cols, n, 0, 1) == KSPLIT, (rows, cols)
    if n < 112:
        assert [plan(t, 5632, 2048, n, 1, 0) for t in (Q4_K, Q5_K)] == [PLANES] * 2
        assert [plan(t, 4096, 14336, n, 0, 1) for t in (Q4_K, Q5_K)] == [PLANES] * 2


@pytest.mark.parametrize("n", [97, 100, 112, 113, 128])
def test_the_fourth_tile_of_32_tokens(plan, n):
    """gate | up of 5632 x 2048 from 97 tokens on: the tiles take as long as at 128, 27 us, the K-split kernel 24."""
    assert [plan(t, 5632, 2048, n, 1, 0) for t in (Q4_K, Q5_K, Q6_K)] == [KSPLIT] * 3


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("n", [161, 180, 212, 256])
def test_the_square_tensor_of_4096_columns(plan, t, n):
    """attn_output of an 8B model from 161 tokens on: 24 to 28 us with the K-split kernel, 17 to 22 on tiles."""
    assert [plan(t, 4096, 4096, n, 0, s) for s in (0, 1)] == [PLANES] * 2
