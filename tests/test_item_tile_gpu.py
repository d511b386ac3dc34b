"""Work items sized by the launch's load: J and K do not depend on how the Q
ranges are cut.  Ranges sized by load are compared with ranges of a fixed
length, from launches with less than one item per wavefront (1 water) to full
ones, in both precisions."""
import numpy
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nwater,basis,precision', [
    (1, 'cc-pvdz', 'fp64'), (2, 'cc-pvtz', 'fp64'), (3, 'def2-svp', 'mixed'),
    (7, 'def2-svp', 'fp64'), (11, 'cc-pvdz', 'mixed')])
@pytest.mark.parametrize('tile', [1, 37])
def test_items_by_load_equal_fixed_items(nwater, basis, precision, tile):
    from byteqc_amd import systems
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf import hf
    lib = load_library()
    mol = systems.water_mole(nwater, systems.box_for_density(nwater) + 1.0, 40 + nwater, basis)
    dm = systems.random_density(mol.nao_nr(), 5 * nwater, 7)
    opt = hf._VHFOpt(mol).build()
    by_load = hf.get_jk(mol, dm, vhfopt=opt, precision=precision)
    flops = hf.last_build_flops()
    try:
        assert lib.BQCset_tile(1, -1, 0, tile) == 0 and lib.BQCset_tile(4, -1, 0, tile) == 0
        fixed = hf.get_jk(mol, dm, vhfopt=opt, precision=precision)
    finally:
        lib.BQCset_tile(0, 0, 0, 0)
    assert numpy.array_equal(flops, hf.last_build_flops())
    # the same quartets added in another order: rounding of sums of ~1e2
    # (J) over at most ~1e4 terms, 1e2 * 2e-16 * sqrt(1e4)
    for a, b in zip(by_load, fixed):
        assert abs(a - b).max() < 1e-11
