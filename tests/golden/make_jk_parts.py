"""J and K of two molecules from the CPU oracle, for tests/test_tile_parts_gpu.py.

``dense``: 14 atoms with one contracted s, p, d and f shell each, large enough
that a build runs the classes of five and six parts in the tile kernel, which
small molecules leave to the wavefront kernel (lower triangles of J and K).
``far``: 70 atoms with one contracted s, p and f shell each, 20 Angstrom apart,
so that only the pairs on one atom are left and 64 neighbouring pairs have 64
different first and second shells (the atoms' blocks of J, the others being
zero, and every 17th row of K).

Run from the repository's root: python -m tests.golden.make_jk_parts (a few
minutes)."""
import os

import numpy

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), 'jk_parts.npz')
K_STEP = 17


def _molecule(shells, xyz):
    from byteqc_amd.gto import M
    basis = [[l] + [[float(e), 1.0 / n] for e in numpy.geomspace(hi, lo, n)]
             for l, n, lo, hi in shells]
    return M(atom=[('H', tuple(r)) for r in xyz], basis={'H': basis})


def dense():
    return _molecule([(0, 4, .3, 3.), (1, 5, .3, 2.), (2, 3, .4, 1.5), (3, 2, .5, 1.2)],
                     [(1.5 * (i % 3), 1.6 * (i // 3 % 2), 1.7 * (i // 6)) for i in range(14)])


def far():
    return _molecule([(0, 5, .3, 3.), (1, 6, .3, 2.), (3, 4, .5, 1.2)],
                     [(20. * (i % 5), 20. * (i // 5 % 4), 20. * (i // 20)) for i in range(70)])


def density(mol):
    from byteqc_amd import systems
    return systems.random_density(mol.nao_nr(), 7, 11)


if __name__ == '__main__':
    from oracle import oracle as orc
    mol = dense()
    j, k = orc.get_jk(mol, density(mol))
    low = numpy.tril_indices(len(j))
    out = dict(dense_j=j[low], dense_k=k[low])
    mol = far()
    j, k = orc.get_jk(mol, density(mol))
    n = len(j) // 70
    blocks = j.reshape(70, n, 70, n)
    out['far_j'] = numpy.stack([blocks[i, :, i] for i in range(70)])
    for i in range(70):
        blocks[i, :, i] = 0
    assert not blocks.any()
    out['far_k'] = k[::K_STEP]
    numpy.savez_compressed(PATH, **out)
