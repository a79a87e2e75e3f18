"""The device's copy of the cache's cell table: a batch uploads only what sequence operations changed and its own set-up launch does not write."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq", [1, 3])
def test_cell_table_follows_sequence_operations(pkg, tmp_path_factory, n_seq):
    """The same calls on two contexts, one of which re-uploads its whole table before every batch (a batch that finds no cells makes the next one do so): rows bit for bit
    the same through cuts of a tail, of the middle and of everything, copies of a sequence, shifts, prompts and steps."""
    path = str(tmp_path_factory.mktemp("cells") / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "tiny-d128", "q4_k_m", seed=3, with_vocab=False)
    m = pkg.Model(path)
    cs = [pkg.Context(m, n_ctx=256, n_batch=512, n_ubatch=512, n_seq_max=n_seq) for _ in range(2)]
    rng = np.random.default_rng(n_seq)
    length = [0] * n_seq

    def batch(s, n):
        toks = rng.integers(0, m.n_vocab, n)
        rows = []
        for k, c in enumerate(cs):
            if k == 1:
                assert c.decode(np.zeros(300, np.int32), np.arange(300) % 200, s) == 1      # more tokens than cells: refused, nothing changes
            assert c.decode(toks, np.arange(length[s], length[s] + n), s) == 0
            rows.append(c.logits())
        length[s] += n
        assert np.array_equal(*rows), (s, n, length)

    for step in range(60):
        s = int(rng.integers(n_seq))
        op = rng.integers(6)
        room = 256 // n_seq - 4 - max(length)
        if length[s] > 4 and (op == 0 or room < 24):
            cut = int(rng.integers(1, length[s]))
            for c in cs:
                c.kv_seq_rm(s, cut, -1)
            length[s] = cut
        elif length[s] > 12 and op == 1:                                                   # a hole, its right side moved over it
            for c in cs:
                c.kv_seq_rm(s, 3, 6)
                c.kv_seq_add(s, 6, -1, -3)
            length[s] -= 3
        elif op == 2 and n_seq > 1:
            d = (s + 1) % n_seq
            for c in cs:
                c.kv_seq_rm(d, -1, -1)
                c.kv_seq_cp(s, d, -1, -1)
            length[d] = length[s]
        elif op == 3 and step % 7 == 0:
            for c in cs:
                c.kv_clear()
            length = [0] * n_seq
        batch(s, 1 if rng.integers(3) else int(rng.integers(2, 20)))
    for c in cs:
        c.close()
    m.close()
