"""A single token's attention over up to four chunks of 64 cells with heads of 64: all of a head's chunks in one workgroup."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_model import FLIP_TOL, KV, be, make, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_seq", [1, 3])                    # by cell count; by the sequence's list of chunks
@pytest.mark.parametrize("cfg,tk,tv", [("tiny-gqa4", "f16", "f16"), ("tiny-gqa4", "q8_0", "q8_0"), ("tiny-gqa4", "q8_0", "f16"), ("tiny-gqa4", "f16", "q8_0"),
                                       ("tiny-tl-2l", "f16", "f16"), ("tiny-tl-2l", "q8_0", "q8_0")])
def test_steps_at_the_edges_of_chunks(be, pkg, tmp_models, cfg, tk, tv, n_seq):  # noqa: F811
    """Four and eight query heads to a kv head, the step's cell the first, the last and one in between of each of the four chunks and of the fifth, where the general form takes over; FLIP_TOL: a
    code of a quantised activation that flips for another order of the sums."""
    path = make(pkg, tmp_models, cfg, "q4_k_m")
    oq.set_fa_v_acc_f32(1 if tv == "f16" else 0)
    try:
        m = pkg.Model(path)
        c = pkg.Context(m, n_ctx=1024, n_seq_max=n_seq, type_k=KV[tk], type_v=KV[tv])
        om = oq.OracleModel(path)
        oc = oq.OracleContext(om, 1024, KV[tk], KV[tv], True, oq.threads())
        toks = np.random.default_rng(7).integers(3, m.n_vocab, 258)
        sq = n_seq - 1
        if sq:                                                # cells of another sequence, which the step must not see
            assert c.decode(toks[:70], np.arange(70), [0] * 70) == 0
        have = 0
        for n in (0, 1, 40, 62, 63, 64, 100, 127, 128, 191, 192, 254, 255, 256, 257):
            if n > have:
                k = n - have
                fl = np.zeros(k, np.int8)
                for x in (c, oc):
                    x.decode(toks[have:n], np.arange(have, n), [sq] * k if x is c else [0] * k, fl)
            assert c.decode([int(toks[n])], [n], [sq], [1]) == 0
            assert rel_err(c.logits(0), oc.decode([int(toks[n])], [n], [0], [1])[0]) <= FLIP_TOL, n
            have = n + 1
        c.close(); m.close(); oc.close(); om.close()
    finally:
        oq.set_fa_v_acc_f32(0)
