"""Single-token steps whose rows nobody reads: they may be queued one behind another, and give the rows that they give one by one."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(pkg, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("queue") / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "tiny-8b-2l", "q4_k_m", seed=6, with_vocab=False)
    m = pkg.Model(path)
    yield m
    m.close()


@pytest.mark.parametrize("n_seq,graphs", [(1, True), (1, False), (2, True)])
def test_unread_steps_give_the_same_rows(pkg, model, n_seq, graphs):
    """Steps, cuts and shifts queued without a read in between against the same calls with the row read after each: the last rows bit for bit, from buckets whose graphs are new
    and from such as have been replayed."""
    rows = []
    for read in (True, False):
        rng = np.random.default_rng(4)
        c = pkg.Context(model, n_ctx=1024, n_batch=512, n_ubatch=512, n_seq_max=n_seq, use_graphs=graphs)
        out, pos = [], [0] * n_seq
        for s in range(n_seq):
            assert c.decode(rng.integers(0, model.n_vocab, 230), np.arange(230), s) == 0      # (the steps below pass 256 cells: another graph)
            pos[s] = 230
        for k in range(60):
            s = int(rng.integers(n_seq))
            if k % 13 == 5:
                c.kv_seq_rm(s, pos[s] - 7, -1)
                pos[s] -= 7
            if k % 17 == 9:
                c.kv_seq_rm(s, 3, 6)
                c.kv_seq_add(s, 6, -1, -3)
                pos[s] -= 3
            assert c.decode([int(rng.integers(model.n_vocab))], [pos[s]], s) == 0
            pos[s] += 1
            if read or k in (30, 59):
                row = c.logits()
                if k in (30, 59):
                    out.append(row)
        c.close()
        rows.append(out)
    for a, b in zip(*rows):
        assert np.isfinite(a).all() and np.array_equal(a, b)


def test_a_step_is_queued_behind_unfinished_work(pkg, model):
    """A step behind a prompt and another step, neither read: its call comes back while the device still works on the prompt."""
    c = pkg.Context(model, n_ctx=4096, n_batch=2048, n_ubatch=2048)
    toks = np.random.default_rng(1).integers(0, model.n_vocab, 2048)
    share = []
    for _ in range(6):
        c.kv_clear()
        assert c.decode(toks, np.arange(2048)) == 0
        assert c.decode([1], [2048]) == 0
        t0 = time.perf_counter()
        assert c.decode([2], [2049]) == 0
        t1 = time.perf_counter()
        c.logits()
        share.append((t1 - t0) / (time.perf_counter() - t0))
    assert min(share[1:]) < 0.5, share                             # (the first pass captures the step's graph)
    c.close()


@pytest.mark.parametrize("n_seq", [1, 2])
def test_first_step_of_a_bucket_and_its_replays(pkg, model, n_seq):
    """A bucket's first step runs by launches, later ones by the graph that was captured behind it: the same token at the same place gives the same row, in the bucket of the
    first 256 cells and in the next."""
    c = pkg.Context(model, n_ctx=1024, n_batch=512, n_ubatch=512, n_seq_max=n_seq)
    rng = np.random.default_rng(8)
    for past in (5, 300):
        c.kv_clear()
        assert c.decode(rng.integers(0, model.n_vocab, past), np.arange(past)) == 0
        rows = []
        for _ in range(4):
            assert c.decode([17], [past]) == 0
            rows.append(c.logits())
            c.kv_seq_rm(0, past, -1)
        assert all(np.array_equal(rows[0], r) for r in rows[1:])
    c.close()
