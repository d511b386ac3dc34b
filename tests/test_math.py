"""Host check of the kernels' scalar arithmetic (byteqc_amd/csrc/bqc_math.h):
reciprocal, quotient and inverse square root round like the exact value, the
factors of a primitive quartet are no less precise than quotients, and the Rys polynomials kept in LDS are no further from the table's exact value
than Clenshaw's rule on the table itself."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope='module')
def errors(tmp_path_factory):
    gxx = shutil.which('g++')
    if gxx is None:
        pytest.skip('no host C++ compiler')
    exe = str(tmp_path_factory.mktemp('math') / 'math_check')
    subprocess.run([gxx, '-std=c++17', '-O2', '-mfma', '-ffp-contract=off', '-o', exe,
                    os.path.join(HERE, 'cpp', 'math_check.cpp')], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    return {n: (float(m), float(r)) for n, m, r in (line.split() for line in out.splitlines())}


@pytest.mark.parametrize('name', ['rcp0', 'div0', 'rsqrt0'])
def test_rounded_like_the_exact_value(errors, name):
    # half a unit in the last place is at most 2^-53 of the value; the long
    # double reference adds 2^-11 of that, a tie decided the other way 2^-12
    assert errors[name][0] <= 1.001


@pytest.mark.parametrize('name', ['a0', 'fac0'])
def test_quartet_factors_no_worse_than_quotients(errors, name):
    # the same number of roundings, some of them halved by the square root:
    # the largest of 2e6 samples differ by a few per cent by chance
    for got, ref in zip(errors[name], errors[f'quotient_{name}']):
        assert got <= 1.05 * ref


@pytest.mark.parametrize('n', range(1, 5))
@pytest.mark.parametrize('f', ['u', 'w'])
def test_rys_rows_no_worse_than_clenshaw(errors, n, f):
    for got, ref in zip(errors[f'{f}{n}'], errors[f'clenshaw_{f}{n}']):
        assert got <= ref
