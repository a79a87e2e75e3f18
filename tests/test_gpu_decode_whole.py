"""A single token's attention over up to four chunks of 64 cells with heads of 64: all of a head's chunks in one workgroup."""
import os
import re
import subprocess
import sys

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


@pytest.mark.parametrize("n_seq", [1, 3])
@pytest.mark.parametrize("cfg,tk,tv", [("tiny-gqa4", "f16", "f16"), ("tiny-gqa4", "q8_0", "f16"), ("tiny-gqa4", "f16", "q8_0"), ("tiny-tl-2l", "f16", "f16"), ("tiny-tl-2l", "q8_0", "q8_0")])
def test_bits_of_the_general_form(be, pkg, tmp_models, cfg, tk, tv, n_seq):  # noqa: F811
    """The same arithmetic in the same order as a workgroup a chunk and their merge behind a ticket: a chunk's sums, the chunks' weights, and the outputs' sum chunk by chunk."""
    m = pkg.Model(make(pkg, tmp_models, cfg, "q4_k_m"))
    toks, out = np.random.default_rng(9).integers(3, m.n_vocab, 258), []
    try:
        for whole in (1, 0):
            be.set_option("attn_whole", whole)
            c = pkg.Context(m, n_ctx=1024, n_seq_max=n_seq, type_k=KV[tk], type_v=KV[tv])
            sq, have, rows = n_seq - 1, 0, []
            if sq:
                assert c.decode(toks[:70], np.arange(70), [0] * 70) == 0
            for n in (0, 1, 2, 31, 63, 64, 65, 127, 128, 130, 191, 192, 230, 254, 255):
                if n > have:
                    assert c.decode(toks[have:n], np.arange(have, n), [sq] * (n - have), np.zeros(n - have, np.int8)) == 0
                assert c.decode([int(toks[n])], [n], [sq], [1]) == 0
                rows.append(c.logits(0).copy())
                have = n + 1
            out.append(np.stack(rows))
            c.close()
    finally:
        be.set_option("attn_whole", 1)
    m.close()
    assert np.array_equal(*out)


PROBED = """
import sys
sys.path.insert(0, %r)
import numpy as np
from __graft_entry__ import load_pkg
pkg = load_pkg()
be = pkg.Backend()
m = pkg.Model(sys.argv[1])
c = pkg.Context(m, n_ctx=512)
n = int(sys.argv[2])
assert c.decode(np.arange(3, 3 + n), np.arange(n)) == 0 and c.decode([5], [n]) == 0
c.close(); m.close()
"""


@pytest.mark.parametrize("n,items", [(100, 4 * 4), (300, 4 * 8)])           # one workgroup's four chunks of each of four kv heads; a workgroup a chunk of 512 cells
def test_probe_reports_either_form(be, pkg, tmp_models, n, items):  # noqa: F811
    """MI355_ATTN_PROBE=1: every item's start and end and the merges' phases, in order."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", PROBED % root, make(pkg, tmp_models, "tiny-tl-2l", "q4_k_m"), str(n)], capture_output=True, text=True, timeout=100, cwd=root,
                       env=dict(os.environ, MI355_ATTN_PROBE="1"))
    assert r.returncode == 0, r.stderr[-2000:]
    got = re.search(r"attn probe: (\d+) workgroups", r.stderr)
    assert got and int(got.group(1)) == items, r.stderr[-2000:]
    merges = re.findall(r"merge: ticket at (\S+) us, weights \+(\S+), sums \+(\S+), stores \+(\S+) -> done at (\S+) us", r.stderr)
    assert len(merges) == 4 and all(0 <= float(x) < 1000 for row in merges for x in row), merges
