"""Batches of 3 .. 8 tokens (csrc/mmq_few.hip): two or four scale groups as rows of one matrix product; 33 .. 48 tokens with the operands in registers; gate | up as eight rows of each."""
import pytest

import test_gpu_few as few
from test_gpu_ops import Q4_K, Q5_K, Q6_K, be  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(2048, 33, 3), (2304, 4113, 4), (11008, 17, 4), (256, 15, 5), (4096, 4130, 8), (5632, 40, 5), (11008, 4112, 8), (4096, 17, 9),      # four, two and one group
                                   (2048, 40, 33), (4096, 4113, 37), (4352, 17, 48)])                                                                                  # one, two and more super-blocks a wave
def test_tokens(be, t, K, N, T):  # noqa: F811
    few.test_few_tokens(be, t, K, N, T)


@pytest.mark.parametrize("types", [(Q4_K, Q4_K, Q6_K), (Q6_K, Q5_K, Q4_K)])
@pytest.mark.parametrize("K,Ns,T", [(4096, (4096, 1024, 1024), 4), (1024, (4096, 4096, 3), 7), (5120, (40, 5, 5), 8), (4096, (6000, 1, 16), 40)])
def test_types_share_the_workgroups(be, types, K, Ns, T):  # noqa: F811
    few.test_tensors_of_one_launch(be, types, K, Ns, T)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(256, 5, 3), (4096, 4100, 4), (11008, 12, 4), (2048, 4097, 8), (5632, 9, 6), (4096, 7, 16), (4096, 4111, 30), (2304, 20, 32), (4352, 4100, 16),
                                   (4096, 4111, 37), (2304, 20, 48), (2048, 9, 33)])         # three token tiles: two super-blocks a wave, all whole and the second ragged; one
def test_gate_up(be, t, K, N, T):  # noqa: F811
    """Fewer rows than a tile of eight, and a last tile that begins among the rows of the one before."""
    few.test_gate_up_pair(be, t, K, N, T)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(4096, 4100, 4), (5632, 31, 7), (4096, 4113, 40)])
def test_residual(be, t, K, N, T):  # noqa: F811
    few.test_residual_on_the_way_out(be, t, K, N, T)
