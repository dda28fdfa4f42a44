"""Which prefill calls run as whole rounds of work-groups and a second launch (host code, at 256 CUs): the shapes
that tests/test_gpu_gemm_rounds.py runs do, the ones measured faster in one launch do not.
"""
import ctypes

import pytest

from oracle_lib import T_Q4_K, T_Q8_0
from test_gpu_gemm_rounds import SHAPES


def _rows(qk, typ, k, n, m):
    fn = qk.lib["_ZN2qk15gemm_round_rowsEiiiimi"]  # int gemm_round_rows(int, int, int, int, size_t, int)
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_size_t, ctypes.c_int]
    return fn(typ, k, n, m, 32 << 20, 256)


@pytest.mark.parametrize("typ,k,n,m", SHAPES, ids=[f"t{t}k{k}n{n}m{m}" for t, k, n, m in SHAPES])
def test_two_launches(qk, typ, k, n, m):
    rows = _rows(qk, typ, k, n, m)
    assert 0 < rows < n and rows % 2048 == 0  # eight groups of eight tile pairs, as that test's seams assume


@pytest.mark.parametrize("typ,k,n,m", [(T_Q4_K, 5120, 17408, 1024), (T_Q4_K, 5120, 17408, 1500), (T_Q4_K, 5120, 17408, 512),
                                       (T_Q8_0, 6144, 5120, 100), (T_Q8_0, 6144, 5120, 64)])
def test_one_launch(qk, typ, k, n, m):
    assert _rows(qk, typ, k, n, m) == 0
