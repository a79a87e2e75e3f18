"""Batches of 3 .. 64 tokens against K-quant weights (csrc/mmq_few.hip): the contraction whose workgroups walk 16-row tiles with the quantiser's operand blocks, and the K-split
kernel of csrc/mmq.hip that takes the other half of these batches: the same integers, the same fold, the same order of f32 sums, so the same bits."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import Q4_K, Q5_K, Q6_K, be, rand_weights  # noqa: F401

pytestmark = pytest.mark.gpu


def both(be, call):  # noqa: F811
    """The call through either kernel."""
    try:
        out = []
        for few in (1, 0):
            be.set_option("mmq_few", few)
            out.append(call())
    finally:
        be.set_option("mmq_few", -1)
    return out


def inputs(rng, types, Ns, K, T):
    return [rand_weights(rng, t, n * K) for t, n in zip(types, Ns)], (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(4096, 40, 4), (256, 8210, 3),       # a few rows; one super-block, more row tiles than workgroups, a ragged last one
                                   (4096, 4200, 16), (2048, 8193, 17),  # a full token tile and one token more; two super-blocks per wave and one, several tiles each
                                   (3584, 4130, 32), (11008, 50, 33),   # super-blocks that do not divide by the waves, up to two and more than two per wave
                                   (1024, 4113, 48), (4096, 17, 49), (5632, 4112, 64)])
def test_few_tokens(be, t, K, N, T):  # noqa: F811
    """Against the oracle: the integer of every super-block is exact and the fold the CPU's, so only the f32 order over super-blocks differs (eight partial sums of
    K / 256 / 8 terms, then eight terms: each f32 rounding is half an ulp, 2e-5 of the largest output as for the other contractions)."""
    rng = np.random.default_rng(5 * K + N + T + t)
    W = rand_weights(rng, t, N * K)
    x = (rng.standard_normal((T, K)) * rng.uniform(0.1, 4.0, (T, 1))).astype(np.float32)
    y, other = both(be, lambda: be.mul_mat(t, W, N, K, x))
    ref = oq.mul_mat(t, W, N, K, x)
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
    assert np.array_equal(y, other)


@pytest.mark.parametrize("types", [(Q4_K, Q4_K, Q6_K), (Q5_K, Q5_K, Q5_K), (Q6_K, Q4_K), (Q6_K, Q6_K, Q6_K)])
@pytest.mark.parametrize("K,Ns,T", [(2048, (4100, 17, 33), 3), (4096, (70, 4130, 1), 16), (3584, (3584, 512, 512), 29), (1280, (40, 40, 8200), 37), (2304, (33, 300, 129), 64)])
def test_tensors_of_one_launch(be, types, K, Ns, T):  # noqa: F811
    """Q | K | V: every tensor of the launch, of its own type and rows, has the bits that it has alone."""
    rng = np.random.default_rng(K + T + sum(types))
    Ns = Ns[:len(types)]
    Ws, x = inputs(rng, types, Ns, K, T)
    y, other = both(be, lambda: be.mul_mat_batch(types, Ws, Ns, K, x))
    for i, (t, n) in enumerate(zip(types, Ns)):
        assert np.array_equal(y[i], other[i])
        assert np.array_equal(y[i], be.mul_mat(t, Ws[i], n, K, x))


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(2048, 4100, 3), (4096, 40, 16), (5632, 4113, 31), (1024, 50, 48), (2304, 4130, 64)])
def test_residual_on_the_way_out(be, t, K, N, T):  # noqa: F811
    """One f32 addition to the product, which is what a product without it gives."""
    rng = np.random.default_rng(K + N + T + t)
    (W,), x = inputs(rng, [t], [N], K, T)
    r = rng.standard_normal((T, N)).astype(np.float32)
    plain = be.mul_mat_batch([t], [W], [N], K, x)[0]
    for y in both(be, lambda: be.mul_mat_batch([t], [W], [N], K, x, resid=r)[0]):
        assert np.array_equal(y, r + plain)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N,T", [(256, 40, 3), (2048, 4100, 16), (3584, 4130, 17), (11008, 50, 32), (2048, 4113, 33), (4096, 17, 49), (1280, 4112, 64)])
def test_gate_up_pair(be, t, K, N, T):  # noqa: F811
    """silu(gate) * up in f32 from the products' bits: expf is within 2 ulp, the sum, the division and the product add three halves (4e-7 of the value); below the smallest
    normal number 1 / (1 + e^-g) may round to zero.  The K-split kernel has the pair to 32 tokens."""
    rng = np.random.default_rng(K + N + T + t)
    Ws, x = inputs(rng, [t, t], [N, N], K, T)
    g, u = (v.astype(np.float64) for v in be.mul_mat_batch([t, t], Ws, [N, N], K, x))
    with np.errstate(over="ignore"):
        ref = g / (1.0 + np.exp(-g)) * u
    be.set_option("mmq_few", 1)
    try:
        y = be.mul_mat_batch([t, t], Ws, [N, N], K, x, swiglu=True)[0]
        assert (np.abs(y - ref) <= 4e-7 * np.abs(ref) + 1e-30 * np.abs(u)).all()
        be.set_option("mmq_few", 0)
        if T <= 32:
            assert np.array_equal(y, be.mul_mat_batch([t, t], Ws, [N, N], K, x, swiglu=True)[0])
        else:
            with pytest.raises(Exception):
                be.mul_mat_batch([t, t], Ws, [N, N], K, x, swiglu=True)
    finally:
        be.set_option("mmq_few", -1)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("K,N", [(1280, 8210), (2048, 4100), (2304, 17), (4096, 40), (11008, 4112), (1024, 50)])
def test_two_tokens(be, t, K, N):  # noqa: F811
    """Against the oracle as in test_few_tokens; from 1280 columns on the bits of the same tokens in a batch of three, below the mat-vec's."""
    rng = np.random.default_rng(K + N + t)
    (W,), x = inputs(rng, [t], [N], K, 3)
    y, ref = be.mul_mat(t, W, N, K, x[:2]), oq.mul_mat(t, W, N, K, x[:2])
    assert np.abs(y - ref).max() <= 2e-5 * np.abs(ref).max() + 1e-6
    if K >= 1280:
        assert np.array_equal(y, be.mul_mat(t, W, N, K, x)[:2])


@pytest.mark.parametrize("ftype", ["q4_k_m", "q5_k_m"])
@pytest.mark.parametrize("kv", [1, 8])
def test_two_tokens_through_a_model(pkg, tmp_path, ftype, kv):
    """Q | K | V, attn_output, gate | up, ffn_down and the head of two tokens: the bits of the same tokens in a batch of three (the attention is columns either way, whose sums are a token's
    own)."""
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, "tiny-e2048", ftype, seed=6, with_vocab=False)
    m = pkg.Model(path)
    toks, out = np.random.default_rng(kv).integers(3, m.n_vocab, 3), []
    for n in (2, 3):
        c = pkg.Context(m, n_ctx=256, n_batch=64, n_ubatch=64, type_k=kv, type_v=kv)
        assert c.decode(toks[:n], np.arange(n), 0, np.ones(n, np.int8)) == 0
        out.append([np.array(c.logits(i)) for i in range(2)] + [np.array([c.argmax(i) for i in range(2)])])
        c.close()
    m.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
