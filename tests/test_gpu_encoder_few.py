"""The encoder's f16 projections (csrc/mmf.hip mmf16_few_kernel): Q | K | V with rope and cache store, attention output, gate | up and down as one launch each."""
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
