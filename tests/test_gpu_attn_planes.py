"""Prompt attention whose V planes are made once for all query tiles and whose chunks reach LDS as they are (csrc/attn_prefill.hip)."""
import numpy as np
import pytest

import oracle_py as oq
from test_gpu_ops import F16, Q8_0, be  # noqa: F401

pytestmark = pytest.mark.gpu


def both(be, tkv, H, G, D, n_cells, T, **options):  # noqa: F811
    """The attention's rows where every tile converts for itself, and with the planes."""
    rng = np.random.default_rng(H * 1000 + n_cells + T)
    kf = (rng.standard_normal((n_cells, G * D)) * 10.0 ** rng.uniform(-3, 0.5, (n_cells, 1))).astype(np.float32)
    vf = (rng.standard_normal((n_cells, G * D)) * 10.0 ** rng.uniform(-5, 3, (n_cells, 1))).astype(np.float32)
    kc, vc = np.stack([oq.quantize(tkv, r) for r in kf]), np.stack([oq.quantize(tkv, r) for r in vf])
    cell_pos = np.arange(n_cells, dtype=np.int32)
    cell_pos[rng.random(n_cells) < 0.1] = -1
    if n_cells > 200: cell_pos[96:160] = -1                                     # whole chunks that nothing sees
    cell_pos[0] = 0
    if options: cell_pos[-1] = n_cells - 1
    q_pos = np.sort(rng.integers(0, n_cells, T)).astype(np.int32)
    q_pos[0], q_pos[-1] = 0, n_cells - 1
    q = rng.standard_normal((T, H, D)).astype(np.float32)
    out = []
    for on in (0, 1):
        for k, v in {**options, "attn_planes": on}.items():
            be.set_option(k, v)
        try:
            out.append(be.flash_attn(q, H, G, D, tkv, kc, tkv, vc, cell_pos, q_pos, 1 / np.sqrt(D)))
        finally:
            for k, v in {"attn_planes": 0, "attn_seqs": 1, "attn_spare": 0}.items():
                be.set_option(k, v)
    return out


@pytest.mark.parametrize("tkv", [Q8_0, F16])
@pytest.mark.parametrize("H,G,D,n_cells,T", [
    (4, 1, 128, 1, 32), (4, 1, 128, 32, 33), (8, 2, 128, 33, 40),               # one cell; a chunk; a chunk of one cell more than that
    (32, 8, 128, 700, 611), (8, 2, 128, 4097, 64),                              # key halves of unequal length; long rows, key splits
    (8, 8, 128, 300, 130), (8, 4, 128, 257, 70), (6, 2, 128, 290, 33), (5, 1, 128, 200, 64), (6, 1, 128, 90, 37), (7, 1, 128, 65, 32), (8, 1, 128, 500, 129),
    (2, 2, 64, 31, 32), (4, 4, 64, 1000, 300), (8, 4, 64, 129, 65), (32, 4, 64, 700, 200), (4, 1, 64, 333, 97)])
def test_the_bits_of_the_tiles_own_conversion(be, tkv, H, G, D, n_cells, T):  # noqa: F811
    """Holes in the cache, ragged tiles and chunks, block scales from subnormal to large: the same integers, scales, halves and order of sums as where every tile converts the chunks it walks."""
    out = both(be, tkv, H, G, D, n_cells, T)
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("tkv", [Q8_0, F16])
@pytest.mark.parametrize("H,G,D,n_cells,T,seqs,spare", [
    (32, 8, 128, 700, 300, 3, 0), (8, 2, 128, 290, 64, 2, 1), (8, 8, 128, 520, 140, 2, 40), (8, 4, 128, 257, 70, 5, 224), (5, 1, 128, 200, 64, 1, 31), (8, 1, 128, 500, 129, 4, 33),
    (32, 4, 64, 700, 200, 2, 255), (4, 4, 64, 300, 150, 1, 45), (8, 4, 64, 129, 65, 3, 97)])
def test_several_conversations_and_a_scan_shorter_than_the_table(be, tkv, H, G, D, n_cells, T, seqs, spare):  # noqa: F811
    """Tiles across two sequences' tokens, cells that some of them share; and cells with positions that lie behind the scanned range, in its last chunk and in whole ones behind it, which
    nothing may see."""
    out = both(be, tkv, H, G, D, n_cells, T, attn_seqs=seqs, attn_spare=spare)
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
    if spare:
        assert not np.array_equal(out[0], both(be, tkv, H, G, D, n_cells, T, attn_seqs=seqs)[0])      # (the spare cells would be seen)
