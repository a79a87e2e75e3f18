"""Kernels that are chosen by the width or number of rows: RMSNorm and quantisation (csrc/act.hip norm_quant_kernel), LayerNorm (layer_norm_wave_kernel), the arg-max of a row and
the router of a mixture of experts (csrc/misc.hip), the embeddings' way to the host."""
import dataclasses

import numpy as np
import pytest

from test_gpu_encoder_few import run
from test_gpu_ops import be  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 7, 31, 32])
@pytest.mark.parametrize("n", [256, 1280, 4096, 4352, 8192, 8448])
def test_rms_norm_widths(be, T, n):  # noqa: F811
    """Rows of one block, ragged rounds of four, held in four and eight loads a thread at most and longer than that; a block a wave and more.  A value passes the roundings of mean, eps,
    root, reciprocal and two products, the root and the reciprocal within two and a half ulps: ten half ulps."""
    rng = np.random.default_rng(n + T)
    x = (rng.standard_normal((T, n)) * 4).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    x64 = x.astype(np.float64)
    ref = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * w
    assert (np.abs(be.rms_norm_mul(x, w, 1e-5) - ref) <= 10 * 2.0 ** -24 * np.abs(ref)).all()


@pytest.mark.parametrize("embd", [256, 768, 1024, 2048, 2304])
@pytest.mark.parametrize("n", [9, 40])
def test_layer_norm_widths(pkg, tmp_path, embd, n):
    """A wave a row with one to eight loads a lane, and the workgroup form behind 2048 columns.  Tolerance as in test_gpu_encoder_few."""
    assert run(pkg, tmp_path, n, n_embd=embd, n_head=embd // 64, n_head_kv=embd // 64, n_ff=512) <= 1.6e-3


@pytest.mark.parametrize("n", [2, 40])
def test_embeddings_of_some_tokens(pkg, tmp_path, n):
    """All tokens flagged (the last norm stores the rows to the host) and all but one (gathered and copied), the one form after the other: the same rows, bit for bit."""
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, dataclasses.replace(pkg.gguf_synth.CONFIGS["nomic-embed-2l"], n_vocab=900), "f16", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=256, n_batch=64, n_ubatch=64)
    toks = np.random.default_rng(n).integers(5, 900, (2, n))
    out = []
    for flags in (np.ones(n, np.int8), np.arange(n) != n // 2, np.ones(n, np.int8)):
        for t in toks:                                       # (a second text over the first one's rows)
            c.kv_seq_rm(0, 0, -1)
            assert c.decode(t, np.arange(n), 0, np.asarray(flags, np.int8)) == 0
            out.append([c.embeddings(i).copy() for i in range(n) if flags[i]])
    full, part, again = out[0:2], out[2:4], out[4:6]
    for f, p, a in zip(full, part, again):
        assert np.array_equal(f, a) and np.array_equal([r for i, r in enumerate(f) if i != n // 2], p)
    assert not np.array_equal(full[0], full[1])
    c.close(); m.close()


@pytest.mark.parametrize("vocab", [900, 901, 33006, 33008, 65539])
def test_arg_max_of_a_row(pkg, tmp_path, vocab):
    """Parts of less than a load a thread and of several rounds, counts that are no multiple of four (single loads)."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tinyllama-1.1b"], n_layer=1, n_vocab=vocab, n_embd=256, n_head=4, n_head_kv=2, n_ff=256)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "q4_k_m", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=64)
    for i, t in enumerate(np.random.default_rng(vocab).integers(3, vocab, 4)):
        assert c.decode([int(t)], [i]) == 0
        assert c.argmax() == int(c.logits(-1).argmax())
    c.close(); m.close()


@pytest.mark.parametrize("experts,used", [(2, 1), (8, 2), (20, 4), (64, 6)])
def test_router_token_by_token_and_in_batches(pkg, tmp_path, experts, used):
    """Steps (the norm within the router's launch), batches of less than 64 tokens (a token a workgroup) and of more (four): the same logits but for codes that flip between
    the kernels of the forms; a token sent to another expert would move them by their own size."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tiny-moe"], n_layer=1, n_expert=experts, n_expert_used=used)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "q4_k_m", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=256, n_batch=128, n_ubatch=128)
    toks = np.random.default_rng(experts).integers(3, 500, 70)
    rows = []
    for size in (1, 35, 70):
        c.kv_seq_rm(0, 0, -1)
        got = []
        for i in range(0, 70, size):
            assert c.decode(toks[i:i + size], np.arange(i, i + size), 0, np.ones(size, np.int8)) == 0
            got += [c.logits(j).copy() for j in range(size)]
        rows.append(np.stack(got).astype(np.float64))
    for r in rows[1:]:
        assert (np.linalg.norm(r - rows[0], axis=1) <= 0.02 * np.linalg.norm(rows[0], axis=1)).all()
    c.close(); m.close()


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("experts,used,K,T,norm", [
    (8, 2, 4096, 1, True), (2, 1, 256, 1, True), (60, 4, 2304, 1, True), (64, 8, 16384, 1, True),          # the norm within; two and one waves to an expert; 64 KB of a row
    (8, 2, 4096, 3, False), (3, 3, 768, 5, False), (64, 6, 16384, 2, False),                                # a token a workgroup
    (8, 2, 4096, 66, False), (5, 2, 8192, 65, False), (64, 4, 256, 64, False),                              # four tokens, the last workgroup's ragged; 128 KB of rows
    (8, 2, 320, 3, False), (8, 2, 16640, 2, False), (4, 1, 8448, 70, False),                                # two launches: columns that are no multiple of 256, rows longer than 64 KB; and 64 rows too long for four
])
def test_router_against_float64(be, f16, experts, used, K, T, norm):  # noqa: F811
    """Products are f32 (f16 weights: of the row's f16 roundings, which numpy makes from the same f32 norm), sums double: half an ulp of every product and of the logit.  Experts are
    compared where the k-th is apart from the next by more than that; the weights follow from the logits, an exponential and two divisions in f32: 1e-6 and twice a logit's error."""
    rng = np.random.default_rng(experts * 1000 + K + T)
    W = (rng.standard_normal((experts, K)) / np.sqrt(K)).astype(np.float16 if f16 else np.float32)
    x = (rng.standard_normal((T, K)) * 3).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, K).astype(np.float32) if norm else None
    lg, ids, w = be.moe_router(1 if f16 else 0, W, x, used, nw, 1e-5)
    if norm:
        mean = np.float32((x * x).astype(np.float64).sum() / K)
        x = (x * (np.float32(1) / np.sqrt(mean + np.float32(1e-5)))) * nw
    x = x.astype(np.float16) if f16 else x
    prod = W.astype(np.float64)[None] * x.astype(np.float64)[:, None]
    ref = prod.sum(-1)
    err = 2.0 ** -24 * (np.abs(prod).sum(-1) + np.abs(ref)) * (4 if norm else 1)          # (the norm: a root and a reciprocal of one ulp each)
    assert (np.abs(lg - ref) <= err).all()
    for t in range(T):
        order = np.argsort(-ref[t], kind="stable")
        gap = ref[t][order][:-1] - ref[t][order][1:]
        if (gap[:used] > 2 * err[t].max()).all() if used < experts else (gap > 2 * err[t].max()).all():
            assert ids[t].tolist() == order[:used].tolist()
        p = np.exp(ref[t][ids[t]] - ref[t].max())
        assert np.allclose(w[t], p / p.sum(), rtol=1e-6 + 2 * err[t].max(), atol=0)
