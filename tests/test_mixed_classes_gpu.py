"""Mixed precision: which classes of a build run in FP32 when the bound lets
every quartet (fp32_cut 1e30), and that the others keep FP64 accuracy."""
import pytest

pytestmark = pytest.mark.gpu


# s and p shells: every class has an FP64 tile kernel, so the build is an FP64
# build (the same sums in another order: some 1e5 terms of rounding 1e-16).
# With d shells (dd|dp) and (dd|dd), the wavefront-kernel classes, take FP32
# (2^-24 = 6e-8 per operation, a few hundred operations per quartet).
@pytest.mark.parametrize('basis,fp32,tol', [
    ([[0, [0.9, 1.0]], [1, [0.8, 1.0]]], set(), 1e-12),
    ([[0, [0.9, 1.0]], [1, [0.8, 1.0]], [2, [1.1, 1.0]]], {2221, 2222}, 1e-5)])
@pytest.mark.parametrize('natom', [2, 9])
def test_fp32_classes(natom, basis, fp32, tol):
    from byteqc_amd import systems
    from byteqc_amd.gto import M
    from byteqc_amd.scf import hf
    mol = M(atom=[('H', (1.7 * (i % 3), 1.9 * (i // 3), 0.1 * i)) for i in range(natom)],
            basis={'H': basis}, spin=natom % 2)
    dm = systems.random_density(mol.nao_nr(), 3, 5)
    j0, k0 = hf.get_jk(mol, dm)
    hf.profile_enable(True)
    try:
        j1, k1 = hf.get_jk(mol, dm, precision='mixed', fp32_cut=1e30)
        used = {r['cls'] for r in hf.profile_read() if r['kind'] & 2 and r['nquart'] > 0}
    finally:
        hf.profile_enable(False)
    assert used == fp32
    assert abs(j1 - j0).max() < tol * abs(j0).max() and abs(k1 - k0).max() < tol * abs(k0).max()
