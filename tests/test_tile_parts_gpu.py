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


# with the bound out of the way a mixed build runs exactly the classes without
# a tile kernel in FP32 (test_jk_gpu.py compares such a build with FP64)
def test_fp32_classes_of_cc_pvtz():
    from byteqc_amd import systems
    from byteqc_amd.scf import hf
    mol = systems.water_mole(1, 4.0, 3, 'cc-pvtz')
    pairs = [(a, b) for a in range(4) for b in range(a + 1)]
    nf = lambda l: (l + 1) * (l + 2) // 2  # noqa: E731
    want = {a * 1000 + b * 100 + c * 10 + d for i, (a, b) in enumerate(pairs)
            for c, d in pairs[:i + 1] if nf(a) * nf(b) * nf(c) * nf(d) > 81} - PARTS
    hf.profile_enable(True)
    try:
        hf.get_jk(mol, systems.random_density(mol.nao_nr(), 5, 2), precision='mixed',
                  fp32_cut=1e30)
        recs = [r for r in hf.profile_read() if r['nquart'] > 0]
    finally:
        hf.profile_enable(False)
    assert {r['cls'] for r in recs if r['kind'] & 2} == want
    assert {r['cls'] for r in recs if not r['kind'] & 2} >= PARTS
