"""ctypes binding of liblcq.so — the only way the Python layer reaches the GPU.

There is deliberately no CPU fallback: if the shared object is missing or a
tensor is not on the GPU, calls raise.
"""
from __future__ import annotations

import ctypes as C
import re
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent
LIB_PATH = _PKG / 'liblcq.so'
HEADER = _PKG.parent / 'include' / 'lcq.h'

# constants mirrored from include/lcq.h
F32, BF16, F16 = 0, 1, 2
CODE_NONE, CODE_U8, CODE_I8, CODE_I32, CODE_SAME, CODE_F32, CODE_FP8, CODE_CT4, CODE_CT8 = range(9)
FLAG_SYM, FLAG_NO_ROUND_ZP, FLAG_STATIC, FLAG_SCALAR_QP = 1, 2, 4, 8
FLAG_TIE_EVEN, FLAG_NO_SUBNORMALS, FLAG_DQ_F32 = 16, 32, 64
FLAG_RANGE_BF16, FLAG_SCALE_F32, FLAG_ROW_QP = 128, 256, 512
FLAG_ROWS16 = 4096
FLAG_RANGE_F16 = 8192
FLAG_PROMOTED, FLAG_SCALES_F16 = 16384, 32768

_ERR = {-1: 'invalid argument', -2: 'misaligned pointer', -3: 'unsupported dtype', -4: 'kernel launch failed',
        -5: 'workspace too small', -6: 'input larger than the entry point\'s stated maximum'}


class LcqError(RuntimeError):
    pass


_lib = None


def _header_text() -> str:
    return '\n'.join(re.sub(r'/\*.*?\*/', '', h.read_text(), flags=re.S) for h in sorted(HEADER.parent.glob('*.h')))


def declared_symbols() -> list[str]:
    """Names of every function the headers under include/ declare (lcq.h: the boundary; lcq_bench.h: benchmark aids)."""
    return sorted(set(re.findall(r'\b(lcq_[a-z0-9_]+)\s*\(', _header_text())))


def _signatures() -> dict:
    """name -> (restype, argtypes) as the headers declare them.  With its argument types known, a foreign function takes
    plain Python numbers and addresses: no ctypes object has to be made per argument (5 us of a call with 14 of them)."""
    simple = {'int': C.c_int, 'int64_t': C.c_int64, 'float': C.c_float}
    out = {}
    for ret, name, params in re.findall(r'\b(int64_t|int)\s+(lcq_[a-z0-9_]+)\s*\(([^)]*)\)\s*;', _header_text()):
        types = []
        for p in (q.strip() for q in params.split(',')):
            if p not in ('', 'void'):
                types.append(C.c_void_p if '*' in p else simple[p.split()[0]])
        out[name] = (simple[ret], types)
    return out


def lib() -> C.CDLL:
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise LcqError(f'{LIB_PATH} is missing: run `python -m lightcompress_amd.build` '
                           '(there is no CPU fallback for this path)')
        handle = C.CDLL(str(LIB_PATH))
        for name, (restype, argtypes) in _signatures().items():
            fn = getattr(handle, name)
            fn.restype, fn.argtypes = restype, argtypes
        _lib = handle
    return _lib


def dtype_code(dt: torch.dtype) -> int:
    if dt == torch.float32:
        return F32
    if dt == torch.bfloat16:
        return BF16
    if dt == torch.float16:
        return F16
    raise LcqError(f'unsupported dtype {dt}')


def ptr(t):
    """Device address of a tensor (None -> NULL)."""
    if t is None:
        return None
    if not t.is_cuda:
        raise LcqError('liblcq operates on GPU tensors only (no CPU fallback)')
    if not t.is_contiguous():
        raise LcqError('tensor must be contiguous')
    return t.data_ptr()


def stream():
    """The current stream of the current device, as an address.  (torch.cuda.current_stream() builds a Stream object
    around the same value: 2.8 us against 0.2.)"""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def check(rc: int, what: str):
    if rc != 0:
        raise LcqError(f'{what} failed: {_ERR.get(rc, rc)} ({rc})')


# argument conversions: what the signatures of the headers take
i64 = i32 = int
f32 = float
