"""The rules by which an entry point takes one of several kernels (csrc/launch_rules.h), over all the forms they accept: compiled with the
host compiler, no GPU needed."""
import ctypes
import itertools
import shutil
import subprocess

import pytest

from lightcompress_amd.build import CSRC

WRAPPERS = '''
#include "launch_rules.h"
extern "C" int rank128(int b_t, long long M, long long N, float alpha, float beta, int in_place, int lower) {
  return (int)lcq::rank128_form(b_t, M, N, alpha, beta, in_place, lower);
}
'''
NONE, SOLVE, WAVES, STREAM = range(4)


@pytest.fixture(scope='module')
def rules(tmp_path_factory):
    if not shutil.which('g++'):
        pytest.skip('no host compiler')
    d = tmp_path_factory.mktemp('rules')
    (d / 'w.cpp').write_text(WRAPPERS)
    subprocess.run(['g++', '-std=c++17', '-shared', '-fPIC', f'-I{CSRC}', str(d / 'w.cpp'), '-o', str(d / 'w.so')], check=True)
    return ctypes.CDLL(str(d / 'w.so'))


def test_products_of_depth_128(rules):
    """Only kernels that leave out the tiles above the diagonal get a call that asks for it, an update in place is left to the general
    kernels, and a solve has 128 columns."""
    rules.rank128.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong, ctypes.c_float, ctypes.c_float, ctypes.c_int, ctypes.c_int]
    for b_t, in_place, lower in itertools.product((0, 1), repeat=3):
        for M, N in itertools.product((1, 16, 17, 1024, 16384, 16385, 1 << 24), (4, 64, 68, 128, 4096)):
            update, product = rules.rank128(b_t, M, N, -1.0, 1.0, in_place, lower), rules.rank128(b_t, M, N, 1.0, 0.0, in_place, lower)
            assert product == (SOLVE if b_t and N == 128 else NONE)
            assert rules.rank128(b_t, M, N, 1.0, 1.0, in_place, lower) == NONE
            small = -(-M // 16) * -(-N // 64) <= 1024
            if in_place:
                assert update == NONE
            elif b_t or small:
                assert update == WAVES
            else:
                assert update == (NONE if lower else STREAM)
