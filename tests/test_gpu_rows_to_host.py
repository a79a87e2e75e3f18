"""Logits and embedding rows in host memory: the launch that stores them there, with rows that start off 16-byte boundaries, and the copy that takes over from 32 MB on."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_vocab,n,to_host", [(515, 1, True), (515, 7, True), (515, 7, False),       # odd rows, a tail of one to three floats; fetched on demand
                                               (32001, 3, True), (32001, 40, False),                   # more floats than the launch's threads
                                               (132003, 64, True)])                                    # 33.8 MB
def test_logits_rows_are_the_devices(pkg, tmp_path, n_vocab, n, to_host):
    """Every row's sorted head and arg-max are taken from the device's row: the host's row must hold exactly these."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tiny"], n_vocab=n_vocab)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "q4_k_m", seed=2, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=256, n_batch=128, n_ubatch=128, logits_to_host=to_host)
    rng = np.random.default_rng(n_vocab + n)
    for start in (0, n):                                          # the second batch's rows take the first one's place
        assert c.decode(rng.integers(0, n_vocab, n), np.arange(start, start + n), 0, np.ones(n, np.int8)) == 0
        for i in range(n):
            row = c.logits(i)
            toks, lg = c.topk(32, i)
            assert np.isfinite(row).all() and c.argmax(i) == int(row.argmax())
            assert np.array_equal(row[toks], lg) and np.array_equal(np.sort(row)[::-1][:32], lg)
    c.close(); m.close()


def test_single_steps_rows_in_a_graph(pkg, tmp_path):
    """An F16 head leaves a step's row to the launch inside the captured graph: every replay's row against the device's."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tiny"], n_vocab=515)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "f16", seed=2, with_vocab=False)
    m = pkg.Model(path)
    c, e = pkg.Context(m, n_ctx=64), pkg.Context(m, n_ctx=64, use_graphs=False)
    for pos in range(6):
        assert c.decode([pos + 3], [pos]) == 0 and e.decode([pos + 3], [pos]) == 0
        row = c.logits()
        toks, lg = c.topk(32)
        assert np.array_equal(row[toks], lg) and np.array_equal(row, e.logits())
    c.close(); e.close(); m.close()
