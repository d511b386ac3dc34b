"""Pair data and passes that get_jk does not choose by itself: contracted pairs
without the records of BQCset_prim_records (a caller of the plain
GINTinit_basis_prod_* interface has none), and the two-pass row kernels of
BQCset_row_split."""
import numpy
import pytest

from .test_ref_abi_gpu import per_task_get_jk

pytestmark = pytest.mark.gpu

# the J/K parity bar of the FP64 kernels against the oracle
TOL = 1e-10


@pytest.mark.parametrize('nwater', [1, 3])
def test_contracted_pairs_without_records(nwater):
    from byteqc_amd import systems
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf import hf
    from oracle import oracle as orc
    mol = systems.water_mole(nwater, 4.0, 21, 'def2-svp')
    dm = systems.random_density(mol.nao_nr(), 5 * nwater, 9)
    opt = hf._VHFOpt(mol).build()
    assert opt.cp_nprim.max() > 1
    assert load_library().BQCset_prim_records(opt.bpcache, None) == 0
    ref = orc.get_jk(mol, dm)
    for got in (hf.get_jk(mol, dm, vhfopt=opt),
                [x.cpu().numpy() for x in per_task_get_jk(mol, dm, opt)]):
        for a, b in zip(got, ref):
            assert abs(a - b).max() < TOL


# the two passes need 2048 Cartesian AOs; the build they are compared with is
# compared with the oracle in test_full_size_gpu.py
def test_two_pass_row_kernels():
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf import hf
    from byteqc_amd.systems import workload
    mol, dm, _ = workload('c2')
    opt = hf._VHFOpt(mol).build()
    lib = load_library()
    ref = hf.get_jk(mol, dm, vhfopt=opt)
    flops = hf.last_build_flops()
    hf.profile_enable(True)
    try:
        assert lib.BQCset_row_split(-1, 1) == 0
        got = hf.get_jk(mol, dm, vhfopt=opt)
        recs = hf.profile_read()
    finally:
        lib.BQCset_row_split(-1, -1)
        hf.profile_enable(False)
    assert numpy.array_equal(flops, hf.last_build_flops())
    # a-side (1) and b-side (9) passes of the s/p/d classes up to 27 components
    split = {0, 1000, 1010, 1100, 1110, 2000, 2010, 2100}
    for kind in (1, 9):
        assert split <= {r['cls'] for r in recs if r['kind'] == kind}
    assert not split & {r['cls'] for r in recs if r['kind'] == 17}
    for a, b in zip(got, ref):
        assert abs(a - b).max() < TOL
