"""A batch's last layer behind its K and V rows works on the flagged rows alone where they follow one another (runtime.cc run_layers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be(pkg):
    return pkg.Backend()


# the attention kernels a part of a batch can come to: the one-token kernel (few tokens), columns, query tiles, the general one (a head size with NEOX pairs and biases); block types of every
# contraction; experts by the mat-vec, by groups and as one launch; a q4_0 cache
MODELS = [("tiny-8b-attn-2l", "q4_k_m", 8), ("tiny-7b-attn-2l", "q5_k_m", 1), ("tiny-tl-2l", "q8_0", 1), ("tiny-d128", "q4_k_m", 2), ("tiny-moe", "q5_k_m", 1), ("tiny-qwen2", "q4_k_m", 8)]
CUT = 4                                                      # Context.batch_route


def model(pkg, tmp_models, cfg, ftype):
    path = tmp_models / ("%s-%s.gguf" % (cfg, ftype))
    if not path.exists():
        pkg.gguf_synth.write_synthetic_llama(str(path), cfg, ftype, seed=11, with_vocab=False)
    return pkg.Model(str(path))


def either_way(be, pkg, m, kv, n, flags):
    """The flagged rows' logits and the row of the step behind them, with theirs alone and with every row worked on."""
    toks = np.random.default_rng(n).integers(0, m.n_vocab, n + 41)
    marks = np.zeros(n, np.int8)
    marks[flags] = 1
    follow = not flags or flags[-1] - flags[0] == len(flags) - 1
    rows, behind = [], []
    try:
        for alone in (1, 0):
            be.set_option("last_rows", alone)
            c = pkg.Context(m, n_ctx=512, n_batch=512, n_ubatch=512, type_k=kv, type_v=kv)
            assert c.decode(toks[:40], np.arange(40)) == 0
            assert c.decode(toks[40:40 + n], np.arange(40, 40 + n), 0, marks) == 0
            assert (c.batch_route()[0] & CUT != 0) == (alone and follow)
            rows.append([c.logits(i).astype(np.float64) for i in flags])
            assert c.decode(toks[-1:], [40 + n]) == 0
            behind.append(c.logits())
            c.close()
    finally:
        be.set_option("last_rows", 1)
    assert np.isfinite(behind[0]).all() and np.array_equal(behind[0], behind[1])                 # the cache is the same either way
    return list(zip(*rows))


@pytest.mark.parametrize("cfg,ftype,kv", MODELS)
@pytest.mark.parametrize("n,flags", [(2, [1]), (20, [19]), (33, [32]), (70, [69]), (300, [299]), (300, [120, 121, 122]), (300, list(range(250, 300))), (45, list(range(3, 44))), (70, []), (20, []),
                                     (70, [3, 69]), (300, [])])
def test_flagged_rows_alone(be, pkg, tmp_models, cfg, ftype, kv, n, flags):
    """Flagged rows of a prompt behind another, with every row worked on and with theirs alone: sums in another order, an int8 rounding that falls the other way here and there in the last layer's
    four products (as between a step and a prompt, 0.019 over eight layers; two and a half times that is allowed).  That every kernel a part can come to is reached; whose rows they are,
    test_the_rows_are_theirs says."""
    m = model(pkg, tmp_models, cfg, ftype)
    for a, b in either_way(be, pkg, m, kv, n, flags):
        assert np.linalg.norm(a - b) <= 0.05 * np.linalg.norm(b), np.linalg.norm(a - b) / np.linalg.norm(b)
    m.close()


# the one-token kernel with chunk lists behind a store of its own (1024 values of K and V a row), columns and query tiles; the general attention and columns where there is no such store; NEOX pairs
@pytest.mark.parametrize("cfg,kv", [("tiny-g8", 8), ("tiny-g8", 1), ("tiny-tl-2l", 1), ("tiny-d128", 8), ("tiny-qwen2", 8)])
@pytest.mark.parametrize("n,flags", [(2, [1]), (20, [19]), (20, [4, 5, 6]), (33, [32]), (70, [69]), (300, [299]), (300, [120, 121, 122])])
def test_the_rows_are_theirs(be, pkg, tmp_models, cfg, kv, n, flags):
    """f16 weights, so that nothing is rounded to int8 behind the cache: a row's products round their input to f16 in either kernel (2.8e-4 of a value at the root mean square, where a kernel for
    more rows does and one for fewer does not) and its sums are in another order: below 1e-3 of the largest logit.  One key more or less of 42 to 340 is a twentieth to a seventh of the attention's
    output."""
    m = model(pkg, tmp_models, cfg, "f16")
    for a, b in either_way(be, pkg, m, kv, n, flags):
        assert np.abs(a - b).max() <= 1e-3 * np.abs(b).max(), np.abs(a - b).max() / np.abs(b).max()
    m.close()


@pytest.mark.parametrize("cfg,ftype,kv,bound", [("tiny-8b-attn-2l", "q4_k_m", 8, 0.05), ("tiny-g8", "f16", 8, 1e-3), ("tiny-g8", "f16", 1, 1e-3), ("tiny-tl-2l", "f16", 1, 1e-3)])
@pytest.mark.parametrize("n", [24, 80])
def test_two_sequences_of_a_batch(be, pkg, tmp_models, cfg, ftype, kv, bound, n):
    """The rows at the end of a batch of two sequences, whose cells lie apart: each sees its own keys.  Bounds as above, of the largest logit."""
    m = model(pkg, tmp_models, cfg, ftype)
    toks = np.random.default_rng(3).integers(0, m.n_vocab, 160)
    seq, pos = np.repeat([0, 1], n // 2), np.tile(np.arange(n // 2), 2)
    order = np.r_[0:n // 2 - 1, n // 2:n - 1, n // 2 - 1, n - 1]                                # both sequences' last tokens behind the others
    marks = np.zeros(n, np.int8)
    marks[-2:] = 1
    rows = []
    try:
        for alone in (1, 0):
            be.set_option("last_rows", alone)
            c = pkg.Context(m, n_ctx=512, n_batch=512, n_ubatch=512, n_seq_max=2, type_k=kv, type_v=kv)
            assert c.decode(toks[:n][order], pos[order], seq[order], marks) == 0
            assert (c.batch_route()[0] & CUT != 0) == bool(alone)
            rows.append([c.logits(n - 2).astype(np.float64), c.logits(n - 1).astype(np.float64)])
            c.close()
    finally:
        be.set_option("last_rows", 1)
    for a, b in zip(*rows):
        assert np.abs(a - b).max() <= bound * np.abs(b).max()
    m.close()
