"""Attention of short batches of one sequence (csrc/attn_cols.hip): (token, head) pairs as the columns of 32-wide tiles, waves and workgroups sharing the keys."""
import dataclasses

import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import F16, Q8_0, be  # noqa: F401
from test_oracle_encoder import bert_forward_f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tkv", [Q8_0, F16])
@pytest.mark.parametrize("H,G,D,n_cells,T,shares", [
    (8, 8, 128, 1, 1, 1), (8, 2, 128, 32, 8, 1), (8, 2, 128, 33, 9, 1),         # one cell; a full tile and chunk; one column tile more, a chunk of one cell
    (32, 8, 128, 129, 5, 1), (4, 4, 64, 300, 33, 1), (32, 4, 64, 257, 3, 1),    # four chunks a workgroup and more than that; eight heads a group
    (6, 2, 128, 70, 21, 1), (14, 2, 128, 200, 11, 3), (24, 8, 64, 90, 7, 1),    # groups whose heads do not divide a tile
    (8, 2, 128, 300, 40, 2), (32, 8, 128, 700, 37, 6), (12, 12, 64, 1000, 64, 5), (4, 2, 64, 100, 50, 4),    # shares, some with fewer chunks than waves
    (8, 2, 128, 300, 70, 2), (4, 4, 128, 90, 65, 1), (12, 12, 64, 200, 66, 1), (8, 1, 64, 700, 130, 3), (12, 4, 64, 150, 67, 1),    # over 64 tokens: pairs of f16; three heads of 64 a group do not go to the prompt kernel
])
def test_against_the_oracle(be, tkv, H, G, D, n_cells, T, shares):  # noqa: F811
    """Holes in the cache, a query that sees one cell, ragged tiles and chunks.  q8_0: the scores' integers are exact; f16: the CPU's sums of V are made in f32 for the comparison.
    What differs is the order of f32 sums over D and over the cells and the device's exp2: 2e-5 of the largest output, as for the prompt kernel."""
    rng = np.random.default_rng(H * 1000 + n_cells + T)
    kf = rng.standard_normal((n_cells, G * D)).astype(np.float32)
    vf = (rng.standard_normal((n_cells, G * D)) * rng.uniform(0.2, 3.0, (n_cells, 1))).astype(np.float32)
    kc, vc = np.stack([oq.quantize(tkv, r) for r in kf]), np.stack([oq.quantize(tkv, r) for r in vf])
    cell_pos = np.arange(n_cells, dtype=np.int32)
    cell_pos[rng.random(n_cells) < 0.1] = -1
    cell_pos[0] = 0
    q_pos = np.sort(rng.integers(0, n_cells, T)).astype(np.int32)
    q_pos[0], q_pos[-1] = 0, n_cells - 1
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    scale = 1 / np.sqrt(D)
    be.set_option("attn_cols", shares)
    try:
        out = be.flash_attn(q, H, G, D, tkv, kc, tkv, vc, cell_pos, q_pos, scale)
    finally:
        be.set_option("attn_cols", 0)
    oq.set_fa_v_acc_f32(1 if tkv == F16 else 0)
    try:
        for i in range(T):
            cells = np.nonzero((cell_pos >= 0) & (cell_pos <= q_pos[i]))[0].astype(np.int32)
            ref = oq.flash_attn(q[i], H, G, D, tkv, kc, tkv, vc, cells, scale)
            assert np.abs(out[i] - ref).max() <= 2e-5 * max(1.0, float(np.abs(ref).max())), (i, np.abs(out[i] - ref).max())
    finally:
        oq.set_fa_v_acc_f32(0)


@pytest.mark.parametrize("tkv", [Q8_0, F16])
@pytest.mark.parametrize("H,G,D,shares", [(8, 2, 128, 1), (8, 2, 128, 3), (8, 1, 64, 1), (8, 8, 64, 2)])
@pytest.mark.parametrize("what", ["small weights", "large values"])
def test_weights_and_values_as_in_f32(be, tkv, H, G, D, shares, what):  # noqa: F811
    """Small weights: every query's largest score, 16 over the others, is a cell's whose values are zero, so the output is the others', of weights near 1e-7.  Large values: up to 3e6 in a
    q8_0 cache (the blocks of a row of very different size, a hidden cell among them), 6e4 in an f16 one.  The bound is of the output's own largest: a score of 16 is 2e-6 off in f32, the
    oracle's sum over 300 cells in f32 about as much, together below 2e-5."""
    n, T = 300, 9
    rng = np.random.default_rng(D + H + shares)
    kf = (0.2 * rng.standard_normal((n, G, D))).astype(np.float32)
    vf = rng.standard_normal((n, G, D)).astype(np.float32)
    q = rng.choice([-1.0, 1.0], D) + 0.05 * rng.standard_normal((T, H, D))
    scale = 1 / np.sqrt(D)
    if what == "small weights":
        kf[40] = np.sign(q[0, 0]) * 16 * scale
        vf[40] = 0.0
    else:
        vf *= 10.0 ** rng.uniform(-3, 4.5 if tkv == F16 else 6, (n, G, 1))
        vf[::7, :, D // 2:] *= 1e-3
        vf = np.clip(vf, -6e4, 6e4) if tkv == F16 else np.clip(vf, -3e6, 3e6)
        vf[77] = 6e4 if tkv == F16 else 3e6
    vf = vf.astype(np.float32)
    kc, vc = np.stack([oq.quantize(tkv, r.reshape(-1)) for r in kf]), np.stack([oq.quantize(tkv, r.reshape(-1)) for r in vf])
    cell_pos = np.arange(n, dtype=np.int32)
    cell_pos[77] = -1
    q, q_pos = q.astype(np.float32), np.linspace(100, n - 1, T).astype(np.int32)
    be.set_option("attn_cols", shares)
    try:
        out = be.flash_attn(q, H, G, D, tkv, kc, tkv, vc, cell_pos, q_pos, scale)
    finally:
        be.set_option("attn_cols", 0)
    oq.set_fa_v_acc_f32(1 if tkv == F16 else 0)
    try:
        for i in range(T):
            ref = oq.flash_attn(q[i], H, G, D, tkv, kc, tkv, vc, np.nonzero((cell_pos >= 0) & (cell_pos <= q_pos[i]))[0].astype(np.int32), scale)
            assert np.abs(out[i] - ref).max() <= 2e-5 * float(np.abs(ref).max()), (i, np.abs(out[i] - ref).max() / np.abs(ref).max())
    finally:
        oq.set_fa_v_acc_f32(0)


@pytest.mark.parametrize("tkv", [Q8_0, F16])
@pytest.mark.parametrize("H,G", [(32, 4), (32, 8), (12, 12)])
@pytest.mark.parametrize("T", [2, 5, 31])
def test_within_one_chunk_against_64_bits(be, tkv, H, G, T):  # noqa: F811
    """Heads of 64 over at most 64 cells: the columns and the general attention, either of which a short batch can come to, are as far from 64 bits.  A weight is a score's exp, whose error is that of
    a sum of 64 products of f32 (2^-24 of it each, in quadrature 8 * 6e-8 of a term, the scores near 1) and an output another sum of up to 64: 5e-7 of the output's norm."""
    D, rng = 64, np.random.default_rng(H * 10 + G + T)
    n = int(rng.integers(T, 65))
    kc, vc = (np.stack([oq.quantize(tkv, r) for r in rng.standard_normal((n, G * D)).astype(np.float32)]) for _ in range(2))
    k, v = (np.stack([oq.dequantize(tkv, r, G * D) for r in rows]).astype(np.float64).reshape(n, G, D) for rows in (kc, vc))
    q = (1.5 * rng.standard_normal((T, H, D))).astype(np.float32)
    qq = np.stack([oq.dequantize(tkv, oq.quantize(tkv, r.reshape(-1)), H * D) for r in q]).astype(np.float64).reshape(T, H, D)
    pos = np.arange(n - T, n, dtype=np.int32)
    s = np.einsum("thd,nhd->thn", qq, np.repeat(k, H // G, 1)) / 8.0
    s[np.broadcast_to(np.arange(n)[None, None, :] > pos[:, None, None], s.shape)] = -np.inf
    w = np.exp(s - s.max(-1, keepdims=True))
    ref = np.einsum("thn,nhd->thd", w / w.sum(-1, keepdims=True), np.repeat(v, H // G, 1))
    try:
        for form in (0, 1):
            be.set_option("attn_cols", form)
            out = be.flash_attn(q, H, G, D, tkv, kc, tkv, vc, np.arange(n, dtype=np.int32), pos, 1 / 8)
            assert np.linalg.norm(out - ref) <= 5e-7 * np.linalg.norm(ref), form
    finally:
        be.set_option("attn_cols", 0)


@pytest.mark.parametrize("kv", [1, 8])
@pytest.mark.parametrize("past,n", [(0, 2), (70, 21), (900, 5), (300, 150)])
def test_a_turn_among_other_conversations(pkg, tmp_path, kv, past, n):
    """A conversation alone, and with its cells dealt out among two others' (chunks of its list that hold their cells, chunks left out): the same sums over the same cells in other
    chunks.  f16 weights, so that only a q8_0 cache rounds in between; a logit's share of a flipped code is below 1e-3 of the largest."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["tinyllama-1.1b"], n_layer=2, n_vocab=900)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "f16", seed=4, with_vocab=False)
    m = pkg.Model(path)
    rng = np.random.default_rng(past + n)
    talk, other = rng.integers(3, 900, past + n), rng.integers(3, 900, 2500)
    out = []
    for alone in (True, False):
        c = pkg.Context(m, n_ctx=4096, n_batch=512, n_ubatch=512, n_seq_max=3, type_k=kv, type_v=kv)
        for i in range(0, past, 45):
            part = talk[i:min(past, i + 45)]
            assert c.decode(part, np.arange(i, i + part.size), 1) == 0
            for s in (() if alone else (0, 2)):
                assert c.decode(other[i:i + 45], np.arange(i, i + 45), s) == 0
        assert c.decode(talk[past:], np.arange(past, past + n), 1) == 0
        out.append(c.logits().copy())
        c.close()
    m.close()
    assert np.abs(out[0] - out[1]).max() <= 1e-3 * np.abs(out[0]).max()


@pytest.mark.parametrize("n", [5, 40, 200])
def test_texts_of_two_sequences_in_one_batch(pkg, tmp_path, n):
    """The encoder with two texts interleaved token by token: tiles whose columns see different cells.  Tolerance as in test_gpu_encoder_few."""
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "nomic-embed-2l", "f16", seed=4, with_vocab=False)
    m = pkg.Model(path)
    c = pkg.Context(m, n_ctx=4096, n_batch=2048, n_ubatch=2048, n_seq_max=2)
    toks = np.random.default_rng(n).integers(5, m.n_vocab, (n, 2))
    assert c.decode(toks.reshape(-1), np.repeat(np.arange(n), 2), [0, 1] * n, np.ones(2 * n, np.int8)) == 0
    got = np.stack([c.embeddings(i) for i in range(2 * n)]).astype(np.float64).reshape(n, 2, -1)
    for s in (0, 1):
        ref = bert_forward_f64(path, toks[:, s], np.arange(n))[-1]
        assert np.linalg.norm(got[:, s] - ref) / np.linalg.norm(ref) <= 1.6e-3
    c.close(); m.close()


@pytest.mark.parametrize("model,past,n", [("tinyllama-1.1b", 0, 2), ("tinyllama-1.1b", 0, 3), ("tinyllama-1.1b", 61, 31), ("tinyllama-1.1b", 200, 2),     # no store of K and V of its own: columns at any size
                                          ("tiny-qwen2", 0, 3), ("tiny-qwen2", 130, 9),                                          # NEOX pairs: so there
                                          ("tiny-d128", 123, 4), ("tiny-d128", 123, 5), ("tiny-d128", 125, 4), ("tiny-d128", 0, 2),      # two chunks of cells, and three
                                          ("tiny-d128-mha", 251, 4), ("tiny-d128-mha", 253, 4), ("tiny-d128-mha", 253, 3)])      # keys of their own: four chunks and five, four tokens and three
@pytest.mark.parametrize("kv", [1, 8])
def test_few_tokens_as_steps(pkg, tmp_path, model, past, n, kv):
    """A few tokens as one batch, on either side of the rule that chooses their kernel, and the same as single steps.  f16 weights: what differs is the order of f32 sums and, of a q8_0
    cache or a rounded activation, a code here and there, whose share of a logit is below 1e-3 of the largest."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS[model], n_layer=2, n_vocab=512)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "f16", seed=5, with_vocab=False)
    m = pkg.Model(path)
    talk = np.random.default_rng(past + n).integers(3, 512, past + n)
    out = []
    for each in (n, 1):
        c = pkg.Context(m, n_ctx=512, n_batch=256, n_ubatch=256, type_k=kv, type_v=kv)
        if past:
            assert c.decode(talk[:past // 2], np.arange(past // 2), 0) == 0 and c.decode(talk[past // 2:past], np.arange(past // 2, past), 0) == 0
        for i in range(past, past + n, each):
            assert c.decode(talk[i:i + each], np.arange(i, i + each), 0) == 0
        if model in ("tinyllama-1.1b", "tiny-qwen2") and each > 1:                                  # (no one-token kernel beside it: by the work, not by the number of cells)
            assert c.batch_route()[0] & 2
        out.append(np.array(c.logits(-1)))
        c.close()
    m.close()
    assert np.abs(out[0] - out[1]).max() <= 1e-3 * np.abs(out[1]).max()
