"""Batched and single-token steps of several conversations: each token's attention walks the 64-cell chunks of its own sequence, also where K and V are stored by the attention launch alone."""
import numpy as np
import pytest

from test_gpu_model import FLIP_TOL, KV, be, make, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ctx", [1024, 512])                # regions of whole chunks; chunks that sequences share
@pytest.mark.parametrize("cfg,kv", [("tiny", "f16"), ("tiny", "q8_0"), ("tiny-tl-2l", "f16"), ("tiny-qwen2", "q8_0"), ("tiny-qwen2-1.5b-2l", "f16"), ("tiny-qwen2-1.5b-2l", "q8_0")])
def test_conversations_against_one_alone(be, pkg, tmp_models, cfg, kv, n_ctx):  # noqa: F811
    """Sequences one short of, at and one past a chunk's end, and of several chunks: ticks of all of them, then single steps in turn, against each alone in a context of its own, where no list
    is kept.  The sums differ in their order; a code that flips for it moves a logit by FLIP_TOL at most."""
    m = pkg.Model(make(pkg, tmp_models, cfg, "q4_k_m"))
    rng = np.random.default_rng(len(cfg) + n_ctx)
    lens = [63, 64, 65, 1, 130, 20]
    toks = [rng.integers(3, m.n_vocab, n + 12).astype(np.int32) for n in lens]
    c = pkg.Context(m, n_ctx=n_ctx, n_seq_max=len(lens), type_k=KV[kv], type_v=KV[kv])
    rows = [[] for _ in lens]
    for s, n in enumerate(lens):
        assert c.decode(toks[s][:n], np.arange(n), seq=[s] * n) == 0
    for i in range(8):
        assert c.decode([int(t[n + i]) for t, n in zip(toks, lens)], [n + i for n in lens], seq=list(range(len(lens))), logits=[1] * len(lens)) == 0
        for s in range(len(lens)):
            rows[s].append(c.logits(s).copy())
    for i in range(8, 12):
        for s, n in enumerate(lens):
            assert c.decode([int(toks[s][n + i])], [n + i], seq=[s]) == 0
            rows[s].append(c.logits().copy())
    c.close()
    for s, n in enumerate(lens):
        c = pkg.Context(m, n_ctx=n_ctx, n_seq_max=1, type_k=KV[kv], type_v=KV[kv])
        assert c.decode(toks[s][:n], np.arange(n)) == 0
        for i in range(12):
            assert c.decode([int(toks[s][n + i])], [n + i]) == 0
            assert rel_err(rows[s][i], c.logits()) <= FLIP_TOL, (s, i)
        c.close()
    m.close()


@pytest.mark.parametrize("cfg,kv", [("tiny-tl-2l", "f16"), ("tiny-qwen2", "q8_0")])
def test_a_single_step_uploads_its_own_list(be, pkg, tmp_models, cfg, kv):  # noqa: F811
    """A lone token among the cells of others walks a list; the counts and that list are uploaded, no others.  Where its sequence holds every chunk there is no list to upload: the launches, and
    the bits, of a context of one sequence."""
    m = pkg.Model(make(pkg, tmp_models, cfg, "q4_k_m"))
    toks = np.random.default_rng(3).integers(3, m.n_vocab, 260)
    rows = []
    for n_seq in (1, 4):
        c = pkg.Context(m, n_ctx=1024, n_seq_max=n_seq, type_k=KV[kv], type_v=KV[kv])
        assert c.decode(toks[:130], np.arange(130)) == 0
        assert c.decode([int(toks[130])], [130]) == 0
        assert c.batch_route() == (0, 0)
        rows.append(c.logits().copy())
        if n_seq > 1:
            assert c.decode(toks[:70], np.arange(70), [2] * 70) == 0
            assert c.decode([int(toks[70])], [70], [2]) == 0
            assert c.batch_route() == (1, 64 + 2)
            assert c.decode([int(toks[131])], [131], [0]) == 0
            assert c.batch_route() == (1, 64 + 3)
        c.close()
    assert np.array_equal(*rows)
    m.close()
