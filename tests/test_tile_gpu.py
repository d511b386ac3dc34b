"""The row kernel with its exchange block in LDS, where its block is smallest,
largest and full: 64 lanes with 64 different shells (the lanes take turns by
halves), Q lists in bin order and in block order, one and two densities, J or K
alone."""
import numpy
import pytest

pytestmark = pytest.mark.gpu

# the J/K parity bar of the FP64 kernels against the oracle
TOL = 1e-10


def _spread_atoms(n, gap):
    from byteqc_amd.gto import M
    basis = {'H': [[0, [0.9, 1.0]], [1, [0.8, 1.0]], [2, [1.1, 1.0]]]}
    side = int(numpy.ceil(n ** (1 / 3)))
    atom = [('H', (gap * (i % side), gap * (i // side % side), gap * (i // side ** 2)))
            for i in range(n)]
    return M(atom=atom, basis=basis)


def _check(mol, tile, n_dm=1, **kw):
    from byteqc_amd import systems
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf import hf
    from oracle import oracle as orc
    lib = load_library()
    dms = numpy.stack([systems.random_density(mol.nao_nr(), 5, 3 + i) for i in range(n_dm)])
    try:
        assert lib.BQCset_tile(1, -1, 0, tile) == 0
        got = hf.get_jk(mol, dms if n_dm > 1 else dms[0], **kw)
    finally:
        lib.BQCset_tile(0, 0, 0, 0)
    for i in range(n_dm):
        ref = orc.get_jk(mol, dms[i])
        for on, a, b in zip((kw.get('with_j', True), kw.get('with_k', True)), got, ref):
            if on:
                assert abs((a[i] if n_dm > 1 else a) - b).max() < TOL


# far atoms: only the pairs on one atom are left, so 64 neighbouring P pairs
# have 64 different first and 64 different second shells; 1, 63, 64, 65 and
# 130 of them.  Tiles of 16 take bin-ordered Q lists, of 64 block-ordered ones.
@pytest.mark.parametrize('natom', [1, 63, 64, 65, 130])
@pytest.mark.parametrize('tile', [16, 64])
def test_distinct_shells_in_every_lane(natom, tile):
    _check(_spread_atoms(natom, 20.0), tile)


# near atoms: every shell pairs with every other
@pytest.mark.parametrize('tile,n_dm,kw', [(16, 1, {}), (64, 2, {}), (200, 1, dict(with_j=False)),
                                          (64, 1, dict(with_k=False))])
def test_all_pairs(tile, n_dm, kw):
    _check(_spread_atoms(12, 1.9), tile, n_dm, **kw)
