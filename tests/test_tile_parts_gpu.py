"""The tile kernel of the larger classes against the oracle: classes in five
and six parts, which only launches with enough work run in it, and f shells
whose rows fill the block (64 lanes with 64 different shells take turns)."""
import numpy
import pytest

from .golden import make_jk_parts as gold

pytestmark = pytest.mark.gpu

# the J/K parity bar of the FP64 kernels against the oracle
TOL = 1e-10
PARTS = {2111, 2120, 2210, 3011, 3110, 3300, 3030, 3020, 3200,   # two
         3021, 3120, 3210, 3111, 3130,                           # five
         2121, 2211, 2220}                                       # six


def _build(mol):
    """J, K and the classes that ran with the tile kernel (kind 17)."""
    from byteqc_amd.scf import hf
    hf.profile_enable(True)
    try:
        jk = hf.get_jk(mol, gold.density(mol))
        recs = [r for r in hf.profile_read() if r['nquart'] > 0]
    finally:
        hf.profile_enable(False)
    return jk, {r['cls'] for r in recs if r['kind'] == 17}


def test_parts():
    (j, k), tile = _build(gold.dense())
    assert PARTS <= tile
    want = numpy.load(gold.PATH)
    low = numpy.tril_indices(len(j))
    assert abs(j[low] - want['dense_j']).max() < TOL
    assert abs(k[low] - want['dense_k']).max() < TOL
    assert abs(j - j.T).max() < TOL and abs(k - k.T).max() < TOL


def test_f_shells_take_turns():
    (j, k), tile = _build(gold.far())
    assert {3000, 3010, 3030, 3130} <= tile
    want = numpy.load(gold.PATH)
    n = len(j) // 70
    blocks = j.reshape(70, n, 70, n).copy()
    for i in range(70):
        assert abs(blocks[i, :, i] - want['far_j'][i]).max() < TOL
        blocks[i, :, i] = 0
    assert not blocks.any()
    assert abs(k[::gold.K_STEP] - want['far_k']).max() < TOL and abs(k - k.T).max() < TOL
