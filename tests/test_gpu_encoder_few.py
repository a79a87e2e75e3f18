"""The encoder's f16 projections (csrc/mmf.hip mmf16_few_kernel): Q | K | V with rope and cache store, attention output, gate | up and down as one launch each."""
import dataclasses

import numpy as np
import pytest

from test_oracle_encoder import bert_forward_f64

pytestmark = pytest.mark.gpu


# fewest tokens the launches take, a full token tile, one token more, ragged tiles, and enough workgroups for two token tiles each (gate | up, then every product)
@pytest.mark.parametrize("n", [8, 32, 33, 187, 705, 1999])
def test_encoder_matches_float64(pkg, tmp_path_factory, n):
    """nomic-embed's geometry (768 and 3072 columns: four and eight waves per product), two layers, two sequences apart, against the graph in 64 bits.  Every product rounds
    its input to f16 (half an ulp: 2.8e-4 of a value at the root mean square of the rounding error), eight products lie one behind the other, LayerNorms keep the scale:
    sqrt(8) * 2.8e-4 = 8e-4; twice that is allowed."""
    path = str(tmp_path_factory.mktemp("enc") / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "nomic-embed-2l", "f16", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=4096, n_batch=2048, n_ubatch=2048, n_seq_max=2)
    rng = np.random.default_rng(n)
    for seq in (0, 1):
        toks = rng.integers(5, m.n_vocab, n)
        assert c.decode(toks, np.arange(n), seq, np.ones(n, np.int8)) == 0
        got = np.stack([c.embeddings(i) for i in range(n)]).astype(np.float64)
        ref = bert_forward_f64(path, toks, np.arange(n))[-1]
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= 1.6e-3, err
    c.close(); m.close()


def run(pkg, tmp_path, n, kv=1, **sizes):
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["nomic-embed-2l"], n_vocab=900, **sizes)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "f16", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=max(256, n), n_batch=n, n_ubatch=n, type_k=kv, type_v=kv)          # (buffers of exactly the batch)
    toks = np.random.default_rng(n).integers(5, m.n_vocab, n)
    assert c.decode(toks, np.arange(n), 0, np.ones(n, np.int8)) == 0
    got = np.stack([c.embeddings(i) for i in range(n)]).astype(np.float64)
    ref = bert_forward_f64(path, toks, np.arange(n))[-1]
    c.close(); m.close()
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("n_ff", [64, 128, 192])
def test_feed_forward_narrower_than_half_the_rows(pkg, tmp_path, n_ff):
    """256 columns and a feed-forward of 64: the f16 rows do not fit its buffers, so the products run one by one; from 128 on they do.  Tolerance as above."""
    assert run(pkg, tmp_path, 40, n_embd=256, n_head=4, n_head_kv=4, n_ff=n_ff) <= 1.6e-3


@pytest.mark.parametrize("n", [40, 700])
def test_eight_waves_for_every_product(pkg, tmp_path, n):
    """1280 columns: Q | K | V with its rope and gate | up with their SwiGLU share K over eight waves; one and two token tiles a workgroup.  Tolerance as above."""
    assert run(pkg, tmp_path, n, n_embd=1280, n_head=20, n_head_kv=20, n_ff=2560) <= 1.6e-3


@pytest.mark.parametrize("n", [33, 187])
def test_cache_in_q8_0(pkg, tmp_path, n):
    """768 columns with a q8_0 cache: Q, K and V as launches of their own, rope and store behind.  A value of a block of 32 is off by up to 1 / 254 of the block's largest, 2.5 to
    3 times its root mean square: 6e-3 of a value at the root mean square of the rounding, in K and in V, through two layers: sqrt(4) * 6e-3 at the most (heads' sums average it)."""
    assert run(pkg, tmp_path, n, kv=8) <= 1.2e-2


# one and two 64-column chunks to every wave, as many columns as are staged at once and more; one token more and less than a tile of 32, and where ffn_down takes two token tiles a
# workgroup for the first time
@pytest.mark.parametrize("n,n_embd,n_ff", [(33, 256, 448), (31, 512, 1088), (341, 768, 3072), (33, 1024, 2048)])
def test_tokens_staged_whole(pkg, tmp_path, n, n_embd, n_ff):
    """Q | K | V and gate | up with a workgroup's token rows whole in LDS (to 768 columns), ffn_down on twelve waves.  Tolerance as above."""
    assert run(pkg, tmp_path, n, n_embd=n_embd, n_head=n_embd // 64, n_head_kv=n_embd // 64, n_ff=n_ff) <= 1.6e-3
