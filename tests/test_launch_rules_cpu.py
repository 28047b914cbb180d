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
extern "C" int panels(int is_static, int has_gidx, int rounded, int group, long long R, long long K, long long i1, int count, long long ldErr,
                      int on16, float qmin, float qmax) {
  return lcq::gptq_by_panels(is_static, has_gidx, rounded, group, R, K, i1, count, ldErr, on16, qmin, qmax);
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


def test_column_blocks_by_panels(rules):
    """Panels take whole aligned blocks whose parameters change at multiples of 16 columns, and not the searched codes of 9 and 10 bits
    that they are slower for; everything else stays with sixteen lanes per row."""
    def panels(is_static=0, gidx=0, rounded=1, group=128, R=4096, K=4096, i1=128, count=128, ldErr=1024, on16=1, bits=4, sym=0):
        lo, hi = (-2.0 ** (bits - 1), 2.0 ** (bits - 1) - 1) if sym else (0.0, 2.0 ** bits - 1)
        c = ctypes.c_longlong
        return bool(rules.panels(is_static, gidx, rounded, group, c(R), c(K), c(i1), count, c(ldErr), on16, ctypes.c_float(lo), ctypes.c_float(hi)))

    for R, sym, bits in itertools.product((1, 64, 1000, 4096, 4097, 28672), (0, 1), (2, 4, 8, 11, 16)):
        for group in (16, 32, 64, 128):
            assert panels(R=R, group=group, bits=bits, sym=sym)
            assert not panels(R=R, group=group, bits=bits, sym=sym, rounded=0)
        for group in (-1, 0, 16, 48, 128, 256):
            assert panels(is_static=1, R=R, group=group, bits=bits, sym=sym)
            assert not panels(is_static=1, gidx=1, R=R, group=group, bits=bits, sym=sym)
        for group in (8, 24, 48, 96, 100, 256):
            assert not panels(R=R, group=group, bits=bits, sym=sym)
    assert not panels(is_static=1, group=8) and not panels(is_static=1, group=100)
    for off in (dict(K=4098), dict(i1=64), dict(count=127), dict(ldErr=1023), dict(on16=0)):
        assert not panels(**off) and not panels(is_static=1, **off)
    # one workgroup of 64 rows or fewer, more than one workgroup per CU of sixteen lanes, short groups, given parameters: panels
    for R, group, bits, sym in itertools.product((16, 64, 256, 4096, 5120), (16, 32, 64, 128), (9, 10), (0, 1)):
        codes, reach = 2 ** bits, 2 ** (bits - 1) if sym else 2 ** bits - 1
        slower = reach <= 512 and codes * group >= 65536 and codes * R > 32768 and R <= 4096
        assert panels(R=R, group=group, bits=bits, sym=sym) == (not slower)
        assert panels(is_static=1, R=R, group=group, bits=bits, sym=sym)
    assert not panels(R=256, bits=9, sym=1) and not panels(R=4096, group=64, bits=10, sym=1)
