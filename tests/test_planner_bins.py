"""Schwarz bins of the task planner: lists in descending log q (bisection) and
in any other order (counting) give the bins of the definition."""
import ctypes

import numpy
import pytest


def _plan(locs, log_q, cond, cutoff, nbins):
    from byteqc_amd.lib import load_library
    from byteqc_amd.scf.hf import _ptr
    ncp = len(locs) - 1
    grp = numpy.zeros((ncp, 2), dtype=numpy.int32)
    nmax = ncp * (ncp + 1) // 2
    cp = numpy.zeros((nmax, 2), dtype=numpy.int32)
    bins = numpy.zeros((nmax, 2 * (nbins + 1)), dtype=numpy.int32)
    dmax = numpy.zeros(nmax)
    nt = ctypes.c_int(0)
    load_library().BQCplan_tasks(ncp, _ptr(grp), _ptr(locs), _ptr(log_q), _ptr(cond), 1, cutoff,
                                 nbins, 1, _ptr(cp), _ptr(bins), _ptr(dmax), ctypes.byref(nt))
    return cp[:nt.value], bins[:nt.value]


@pytest.mark.parametrize('nbins', [1, 10, 33])
@pytest.mark.parametrize('sizes', [(1,), (0, 3), (64, 65, 1000)])
@pytest.mark.parametrize('dmax', [1e-9, 1.0, 37.5])
def test_bins_sorted_and_unsorted(nbins, sizes, dmax):
    rng = numpy.random.default_rng(nbins + len(sizes))
    cutoff = 1e-13
    locs = numpy.append(0, numpy.cumsum(sizes)).astype(numpy.int32)
    lists = [numpy.sort(rng.uniform(-32, 0, n))[::-1] for n in sizes]
    for x in lists:
        x[:len(x) // 5] = 0.0     # clipped bounds, equal values
    cond = numpy.array([[dmax]])
    scale = nbins / numpy.log(min(cutoff / dmax, .1))
    for shuffle in (False, True):
        per = [rng.permutation(x) if shuffle else x for x in lists]
        cp, bins = _plan(locs, numpy.ascontiguousarray(numpy.concatenate(per)), cond, cutoff, nbins)
        for (a, b), row in zip(cp, bins):
            for t, got in ((a, row[:nbins + 1]), (b, row[nbins + 1:])):
                s = numpy.floor(scale * lists[t])
                want = [0] + [int((s < k + 1).sum()) for k in range(nbins)]
                assert list(got) == want
