"""The side streams of a device: one set, whatever the number of streams that
builds are made on, lent to one build at a time."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

# rounding of sums of ~1e2 in another order
TOL = 1e-11


def _system(nwater, basis, seed):
    from byteqc_amd import systems
    from byteqc_amd.scf import hf
    mol = systems.water_mole(nwater, systems.box_for_density(nwater) + 1.0, seed, basis)
    dm = torch.as_tensor(systems.random_density(mol.nao_nr(), 5 * nwater, seed), device='cuda')
    return mol, dm, hf._VHFOpt(mol).build()


def test_one_set_for_all_streams():
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf import hf
    mol, dm, opt = _system(2, 'def2-svp', 80)
    ref = hf.get_jk(mol, dm, vhfopt=opt)
    # kept, so that no two have one handle (torch hands out 32 in turn)
    streams = [torch.cuda.Stream() for _ in range(12)]
    got = [hf.get_jk(mol, dm, vhfopt=opt, return_device=True, stream=s) for s in streams]
    torch.cuda.synchronize()
    for jk in got:
        for a, b in zip(jk, ref):
            assert abs(a.cpu().numpy() - b).max() < TOL
    assert load_library().BQCside_streams() == 3


# builds above 1e11 FLOPs plan, stage and launch their classes in turn: the one
# that has the set on its stream and the side streams, the other beside it on
# its own stream; smaller builds keep one work list
@pytest.mark.parametrize('nwater', [(24, 24), (24, 6)])
def test_class_by_class_builds_on_two_streams_and_threads(nwater):
    from byteqc_amd.scf import hf
    systems_ = [_system(n, 'def2-svp', 90 + i) for i, n in enumerate(nwater)]
    ref, flops = [], []
    for m, d, o in systems_:
        ref.append(hf.get_jk(m, d, vhfopt=o))
        flops.append(hf.last_build_flops().sum())
    assert [f > 1e11 for f in flops] == [n > 6 for n in nwater]
    torch.cuda.synchronize()
    got = [None, None]

    def work(i):
        m, d, o = systems_[i]
        st = torch.cuda.Stream()
        for _ in range(4):   # back to back: the work lists' slots are reused
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
