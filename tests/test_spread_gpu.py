"""A build's launches run next to each other on several streams: whatever
follows on the caller's stream sees all of them, builds of several streams and
threads do not disturb each other, and a graph replayed with other work in
between gives the eager result."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(nwater, basis, seed):
    from byteqc_amd import systems
    from byteqc_amd.scf import hf
    mol = systems.water_mole(nwater, systems.box_for_density(nwater) + 1.0, seed, basis)
    dm = torch.as_tensor(systems.random_density(mol.nao_nr(), 5 * nwater, seed), device='cuda')
    return mol, dm, hf._VHFOpt(mol).build()


# rounding of sums of ~1e2 in another order
TOL = 1e-11


@pytest.mark.parametrize('nwater,basis', [(1, 'cc-pvdz'), (2, 'cc-pvtz'), (6, 'def2-svp')])
def test_builds_on_two_streams_and_threads(nwater, basis):
    from byteqc_amd.scf import hf
    systems_ = [_system(nwater, basis, 60 + i) for i in range(2)]
    ref = [hf.get_jk(m, d, vhfopt=o) for m, d, o in systems_]
    torch.cuda.synchronize()
    got = [None, None]

    def work(i):
        m, d, o = systems_[i]
        st = torch.cuda.Stream()
        for _ in range(4):   # back to back: the work list's two slots are reused
            got[i] = hf.get_jk(m, d, vhfopt=o, return_device=True, stream=st)
        st.synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for i in range(2):
        for a, b in zip(got[i], ref[i]):
            assert abs(a.cpu().numpy() - b).max() < TOL


def test_replayed_branches_equal_eager():
    from byteqc_amd.scf.batch import BatchJK
    sys3 = [_system(n, 'def2-svp', 70 + n) for n in (1, 3, 5)]
    dms = [d for _, d, _ in sys3]
    bj = BatchJK([m for m, _, _ in sys3], vhfopts=[o for _, _, o in sys3])
    ref = [tuple(x.clone() for x in jk) for jk in bj.build(dms)]
    bj.capture(dms)
    for _ in range(4):
        out = bj.replay()
        torch.cuda.synchronize()
        for jk, want in zip(out, ref):
            for a, b in zip(jk, want):
                assert float((a - b).abs().max()) < TOL
        torch.randn(512, 512, device='cuda') @ torch.randn(512, 512, device='cuda')
