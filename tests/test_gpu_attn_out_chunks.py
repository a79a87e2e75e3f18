"""The one-launch attention + attn_output (csrc/attn_out.hip) with a query head to every kv head: items of 64 to 256 cells, by how many a CU would get."""
import dataclasses

import numpy as np
import pytest

from test_gpu_model import FLIP_TOL, be, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [1, 8])
@pytest.mark.parametrize("past", [(3, 255, 511), (512, 700, 1023), (1024, 1278, 1535), (1536, 2047, 2048, 2303)])
def test_items_of_each_size(be, pkg, tmp_path, kv, past):  # noqa: F811
    """First and last cells of the ranges of 64, 128, 192 and 256 cells an item (256 CUs, 32 heads) and of two items a CU, against the two launches: the sums differ in their order, and a code
    of attn_output's input that flips for it moves a logit by FLIP_TOL at most; most steps agree to round-off."""
    path = str(tmp_path / "m.gguf")
    cfg = dataclasses.replace(pkg.gguf_synth.CONFIGS["llama-2-7b"], n_layer=1, n_vocab=300, n_ff=512)
    pkg.gguf_synth.write_synthetic_llama(path, cfg, "q5_k_m", seed=4, with_vocab=False)
    toks = np.random.default_rng(past[-1]).integers(3, 300, past[-1] + 1)
    rows = []
    for fused in (1, 0):
        be.set_option("attn_out_fused", fused)
        try:
            m = pkg.Model(path)
            c = pkg.Context(m, n_ctx=2560, n_batch=512, n_ubatch=512, n_seq_max=1, type_k=kv, type_v=kv)
            out, have = [], 0
            for n in past:
                for i in range(have, n, 512):
                    assert c.decode(toks[i:min(n, i + 512)], np.arange(i, min(n, i + 512))) == 0
                assert c.decode([int(toks[n])], [n]) == 0
                out.append(c.logits().copy())
                have = n + 1
            rows.append(out)
            c.close(); m.close()
        finally:
            be.set_option("attn_out_fused", -1)
    errs = np.array([rel_err(a, b) for a, b in zip(*rows)])
    assert errs.max() <= FLIP_TOL and np.median(errs) <= 1e-5, errs
