"""Prompt contraction in 128-row x 256-token workgroup tiles (csrc/mmq.hip mmq_planes2_kernel): how a batch's 32-token tiles are dealt to workgroups and to their halves."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import Q2_K, Q4_K, Q5_K, Q6_K, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q2_K])
@pytest.mark.parametrize("K,N,T", [(768, 130, 32), (256, 96, 64), (1024, 33, 90),        # a half without tokens; one tile each; two and one, the last one ragged
                                   (768, 160, 128), (512, 70, 160), (768, 128, 224),      # two and two, three and two, four and three
                                   (1280, 129, 250), (768, 256, 256), (512, 40, 257),     # a full half beside a ragged one; both full; nine tiles over two workgroups
                                   (256, 130, 611)])                                      # twenty tiles over three
def test_token_tiles(be, t, K, N, T):  # noqa: F811
    """Against the oracle (f32 order over super-blocks, each rounding half an ulp: 2e-5 of the largest output as for the other contractions) and bit for bit against the
    kernel whose waves take two token tiles: same integers, same fold, same order."""
    rng = np.random.default_rng(5 * K + N + T + t)
    W = rand_weights(rng, t, N * K)
    x = (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)
    be.set_option("mmq_planes", 1)
    be.set_option("mmq_ksplit", 0)
    try:
        be.set_option("mmq_tiles", 4)
        be.set_option("mmq_split", 1)
        y = be.mul_mat(t, W, N, K, x)
        be.set_option("mmq_tiles", 2)
        y2 = be.mul_mat(t, W, N, K, x)
    finally:
        be.set_option("mmq_tiles", 0)
        be.set_option("mmq_split", 0)
        be.set_option("mmq_ksplit", 1)
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
    assert np.array_equal(y, y2)


@pytest.mark.parametrize("t", [Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(2048, 1030, 129), (4096, 516, 300), (1024, 4100, 700), (768, 260, 1040)])
def test_split_by_rule(be, t, K, N, T):  # noqa: F811
    """No tile or split set: K is split by the number of workgroups (four parts, two, none) - or not, below eight super-blocks."""
    rng = np.random.default_rng(3 * K + N + T + t)
    W = rand_weights(rng, t, N * K)
    x = (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)
    be.set_option("mmq_ksplit", 0)
    try:
        y = be.mul_mat(t, W, N, K, x)
    finally:
        be.set_option("mmq_ksplit", 1)
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6


@pytest.mark.parametrize("cfg,n", [("tiny-e2048", 130), ("tiny-e2048", 300), ("tiny-8b-attn-2l", 611), ("tiny-tl-2l", 511)])
def test_partial_sums_left_to_the_norm(pkg, tmp_path, cfg, n):
    """attn_output and ffn_down split K two to four ways and the next norm adds the parts to the residual: a prompt in one batch against the same prompt in batches of
    100 tokens, which take a kernel that splits nothing.  The sums differ in f32 order only - until that flips an int8 code of an activation or a cache row, which moves
    these models' logits by up to 1e-2 (3e-2: the tolerance of the other two-path tests)."""
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "q4_k_m", seed=5, with_vocab=False)
    m = pkg.Model(path)
    toks = np.random.default_rng(n).integers(0, m.n_vocab, n)
    rows = []
    for step in (n, 100):
        c = pkg.Context(m, n_ctx=1024, n_batch=1024, n_ubatch=1024)
        for i in range(0, n, step):
            assert c.decode(toks[i:i + step], np.arange(i, min(i + step, n))) == 0
        rows.append(c.logits().copy())
        c.close()
    m.close()
    assert np.isfinite(rows[0]).all() and np.abs(rows[0] - rows[1]).max() <= 3e-2 * np.abs(rows[1]).max()


@pytest.mark.parametrize("parts", [2, 3, 4])
@pytest.mark.parametrize("cfg,kv,n_rot", [("tiny-8b-attn-2l", 8, 128), ("tiny-7b-attn-2l", 1, 128), ("tiny-8b-attn-2l", 1, 64)])
def test_partial_sums_by_whichever_launch(be, pkg, tmp_path, cfg, kv, n_rot, parts):  # noqa: F811
    """Two, three and four parts of Q | K | V, attn_output and ffn_down, added by the rope + cache store and the norms or by a launch of their own: the same order, so the same
    bits - in the prompt's last row and, through the cache, in a step's behind it.  q8_0 and f16 caches, kv heads as many as query heads, half a head rotated."""
    path = tmp_path / "m.gguf"
    pkg.gguf_synth.write_synthetic_llama(str(path), cfg, "q4_k_m", seed=5, with_vocab=False)
    raw = bytearray(path.read_bytes())
    at = raw.index(b"llama.rope.dimension_count") + len(b"llama.rope.dimension_count")
    assert int.from_bytes(raw[at:at + 4], "little") == 4 and int.from_bytes(raw[at + 4:at + 8], "little") == 128       # (a u32, the head size)
    raw[at + 4:at + 8] = n_rot.to_bytes(4, "little")
    path.write_bytes(raw)
    m = pkg.Model(str(path))
    toks = np.random.default_rng(parts).integers(0, m.n_vocab, 300)
    rows = []
    be.set_option("mmq_split", parts)
    try:
        for late in (1, 0):
            be.set_option("late_sums", late)
            c = pkg.Context(m, n_ctx=512, n_batch=512, n_ubatch=512, type_k=kv, type_v=kv)
            assert c.decode(toks, np.arange(300)) == 0
            rows.append([c.logits()])
            assert c.decode([7], [300]) == 0
            rows[-1].append(c.logits())
            c.close()
    finally:
        be.set_option("mmq_split", 0)
        be.set_option("late_sums", 1)
    m.close()
    assert np.isfinite(rows[0]).all() and np.array_equal(rows[0], rows[1])
