"""Single-token steps of Q8_0 files (csrc/mmvq_stream.hip): from 4 MB on a launch of Q8_0 tensors is a weight stream, attn_output with its input's quantisation in front."""
import dataclasses

import numpy as np
import pytest

from test_gpu_model import be  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,changes", [("tinyllama-1.1b", {}),                     # the size it was measured at: three launches a layer stream
                                         ("tinyllama-1.1b", {"n_ff": 1792}),         # an ffn_down below the line
                                         ("llama-3-8b", {"n_ff": 2048})])            # two passes of columns, heads of 128
def test_bits_of_the_register_ring(be, pkg, tmp_path, cfg, changes):  # noqa: F811
    path = str(tmp_path / "m.gguf")
    pkg.gguf_synth.write_synthetic_llama(path, dataclasses.replace(pkg.gguf_synth.CONFIGS[cfg], n_layer=2, n_vocab=500, **changes), "q8_0", seed=4, with_vocab=False)
    toks = np.random.default_rng(3).integers(3, 500, 60)
    rows = []
    for stream in (1, 0):
        be.set_option("mmvq_stream", stream)
        try:
            m = pkg.Model(path)
            c = pkg.Context(m, n_ctx=256)
            assert c.decode(toks[:50], np.arange(50)) == 0
            out = []
            for i in range(50, 60):
                assert c.decode([int(toks[i])], [i]) == 0
                out.append(c.logits().copy())
            rows.append(np.stack(out))
            c.close(); m.close()
        finally:
            be.set_option("mmvq_stream", 1)
    assert np.array_equal(rows[0], rows[1])
