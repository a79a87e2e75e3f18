"""Logits of several rows (csrc/mmq_few.hip mmq_few_head_kernel): stored to the host while the weights stream, with each row's arg-max."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ftype,embd,vocab", [("q4_k_m", 512, 900), ("q4_k_m", 2048, 33007), ("q5_k_m", 4096, 6151), ("q4_k_m", 5120, 4100)])
def test_rows_and_arg_max(pkg, tmp_path, ftype, embd, vocab):
    """The rows are those of a batch that flags more rows than the launch takes (the K-split kernel and a copy behind it: the same sums in the same order), bit for bit.  Fewer row
    tiles than workgroups, one tile and several runs of them each, a last tile of seven rows; one, two and more super-blocks a wave; one and two token tiles, full and ragged."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tinyllama-1.1b"], n_layer=1, n_vocab=vocab, n_embd=embd, n_head=embd // 64, n_head_kv=embd // 512, n_ff=512)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, ftype, seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=256, n_batch=64, n_ubatch=64, n_seq_max=1)
    toks = np.random.default_rng(vocab).integers(3, vocab, 36)

    def rows(n):
        c.kv_seq_rm(0, 0, -1)
        assert c.decode(toks, np.arange(36), 0, np.array([i < n for i in range(36)], np.int8)) == 0
        return np.stack([c.logits(i) for i in range(n)]), [c.argmax(i) for i in range(n)]

    want, best = rows(36)
    assert best == [int(r.argmax()) for r in want]
    for n in (3, 16, 17, 32, 8, 4):                          # (the ticket is taken anew by every launch)
        got, top = rows(n)
        assert np.array_equal(got, want[:n]) and top == best[:n]
    c.close(); m.close()
