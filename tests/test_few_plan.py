"""The few-token GEMM's plan (csrc/qk_few.hip few_plan, host code: no GPU needed), at 256 CUs: its K-slices stay
among those measured within 5 % of the fastest, and its LDS within a CU's.
"""
import ctypes

import pytest

from oracle_lib import T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0

TYPES = [T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0]
IDS = ["q4k", "q5k", "q6k", "q8_0"]
I, P = ctypes.c_int, ctypes.c_void_p


class FewParams(ctypes.Structure):  # csrc/qk_internal.h
    _fields_ = [("w", P * 4), ("y", P * 4), ("n", I * 4), ("tile0", I * 5), ("cnt", I), ("ntiles", I), ("nsb", I), ("k", I),
                ("m", I), ("x", P), ("xperm", I), ("slices", I), ("wgs", I), ("waves", I), ("lds_ring", I)]


def _plan(qk, typ, k, ns, m, pair=False, cap=32 << 20):
    fn = qk.lib["_ZN2qk8few_planEiRNS_9FewParamsEimmbRm"]  # bool few_plan(int, FewParams&, int, size_t, size_t, bool, size_t&)
    fn.restype = ctypes.c_bool
    fn.argtypes = [I, ctypes.POINTER(FewParams), I, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_bool,
                   ctypes.POINTER(ctypes.c_size_t)]
    p, lds = FewParams(ntiles=sum(ns) // 16, nsb=k // 256, k=k, m=m, cnt=len(ns)), ctypes.c_size_t()
    return (p, lds.value) if fn(typ, p, 256, sum(ns), cap, pair, ctypes.byref(lds)) else (None, 0)


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
@pytest.mark.parametrize("k,n,m,near", [(7168, 512, 5, (4,)), (8192, 512, 5, (4,)), (8192, 512, 13, (4,)), (11264, 512, 5, (3, 4)),
                                        (17408, 512, 5, (3, 4)), (5120, 1024, 5, (2, 3, 4)), (1024, 3072, 5, (4,)),
                                        (3072, 3072, 5, (2, 3, 4)), (3072, 3072, 13, (2, 3, 4))])
def test_pair_slices(qk, typ, k, n, m, near):
    """A pair's second launch reads every slice's parts: few slices, also where k has many super-blocks."""
    p, _ = _plan(qk, typ, k, [n, n], m, pair=True)
    assert p.slices in near, p.slices


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
def test_plans_fit(qk, typ):
    """Any shape: the image and the rings fit the LDS, the slices the partials, the grid the CUs."""
    for k in (256, 1024, 2816, 5120, 17408, 65536):
        for ns in ([16], [512], [5120], [17408, 17408], [12288, 1024, 1024], [248320]):
            for m in (5, 8, 9, 16):
                for cap in (1 << 20, 32 << 20):
                    p, lds = _plan(qk, typ, k, ns, m, pair=len(ns) == 2, cap=cap)
                    if p is None:
                        continue
                    assert lds <= 160 * 1024 and p.waves in (8, 12) and 1 <= p.slices * p.wgs <= 256
                    assert p.wgs <= p.ntiles and p.slices <= k // 256
                    assert (p.slices == 1 and len(ns) != 2) or p.slices * m * sum(ns) <= cap


@pytest.mark.parametrize("typ,k,n,m,few", [(T_Q4_K, 4096, 65536, 16, False), (T_Q4_K, 8192, 128256, 9, False), (T_Q8_0, 3072, 65536, 12, False),
                                           (T_Q4_K, 4096, 65536, 8, True), (T_Q4_K, 3072, 65536, 16, True),
                                           (T_Q4_K, 4096, 151936, 16, True), (T_Q5_K, 4096, 65536, 16, True),
                                           (T_Q6_K, 5120, 248320, 13, True)])
def test_whole_gemm_rounds(qk, typ, k, n, m, few):
    """Q4_K and Q8_0 beyond eight tokens leave calls that fill whole rounds of the GEMM's work-groups to it."""
    assert (_plan(qk, typ, k, [n], m)[0] is not None) == few
