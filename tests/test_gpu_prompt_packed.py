"""Prompt contraction whose Q4_K weights come as codes and Q5_K ones as a byte and a nibble (csrc/mmq.hip mmq_pack_kernel): the ends of their range, and launches of several forms."""
import numpy as np
import pytest

import np_twin as tw
import oracle_py as oq
from test_gpu_ops import BB, Q4_K, Q5_K, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q5_K])
@pytest.mark.parametrize("K,N,T", [(256, 33, 33), (1280, 64, 65), (512, 130, 97), (2048, 40, 300)])
def test_largest_codes_and_scales(be, t, K, N, T):  # noqa: F811
    """Codes, scales and activations at their largest, row by row of another sign or half: every kernel makes the same integers of them, so tiles of either size give the same bits;
    the f32 order over super-blocks is all that is left to the oracle (2e-5 of the largest output, as for random weights)."""
    W = np.zeros(N * K // 256 * BB[t], np.uint8)
    blk = W.view(tw.DT[t]).reshape(N, K // 256)
    blk["d"] = np.float16(1e-2)
    blk["dmin"] = np.float16(1e-2)
    for r in range(N):
        blk["scales"][r] = (0xff, 0x3f, 0xc0, 0x77)[r % 4]
        blk["qs"][r] = (0xff, 0x0f, 0xf0)[r % 3]
        if t == Q5_K:
            blk["qh"][r] = (0xff, 0x55, 0x00)[(r // 2) % 3]
    x = np.ones((T, K), np.float32) * (1.0 + np.arange(T, dtype=np.float32)[:, None])
    x[1::3] *= -1.0
    x[2::3, ::2] *= -1.0
    be.set_option("mmq_ksplit", 0)
    try:
        y = []
        for tiles in (1, 2, 4):
            be.set_option("mmq_tiles", tiles)
            be.set_option("mmq_split", 1)
            y.append(be.mul_mat(t, W, N, K, x))
    finally:
        be.set_option("mmq_tiles", 0)
        be.set_option("mmq_split", 0)
        be.set_option("mmq_ksplit", 1)
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y[2] - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
    assert np.array_equal(y[2], y[0]) and np.array_equal(y[2], y[1])


@pytest.mark.parametrize("ftype", ["q4_k_s", "q4_k_m", "q5_k_m"])
@pytest.mark.parametrize("n", [270, 389])
def test_forms_of_one_launch(be, pkg, tmp_path, ftype, n):  # noqa: F811
    """Q | K | V with an attn_v of another form (Q5_K beside Q4_K, Q6_K beside either) is one launch of the tiles; unsplit, it has the bits of the kernels that take a tensor each."""
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "tiny-8b-attn-2l", ftype, seed=n, with_vocab=False)
    m = pkg.Model(path)
    toks = np.random.default_rng(n).integers(0, m.n_vocab, n)
    rows = []
    be.set_option("mmq_split", 1)
    try:
        for lds in (1, 0):
            be.set_option("mmq_lds_form", lds)
            c = pkg.Context(m, n_ctx=512)
            assert c.decode(toks, np.arange(n)) == 0
            rows.append(c.logits().copy())
            c.close()
    finally:
        be.set_option("mmq_lds_form", -1)
        be.set_option("mmq_split", 0)
    m.close()
    assert np.isfinite(rows[0]).all() and np.array_equal(rows[0], rows[1])
