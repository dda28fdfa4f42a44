"""The int8 GEMV's plan (qk_gemv_plan launches nothing, so this runs without a GPU, at 256 CUs): the
K-slices and the waves of a call.
"""
import pytest

from oracle_lib import T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0

TYPES = [T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0]
IDS = ["q4k", "q5k", "q6k", "q8_0"]
FAKE, INT8 = 1 << 20, 1  # an aligned address that nothing reads; QK_GEMV_INT8


def _plan(qk, typ, k, ns, m, glu=False, **knobs):
    try:
        for name, v in knobs.items():
            qk.set_tuning(name, v)
        return qk.gemv_plan([qk.weight_view(FAKE, typ, k, n, 1) for n in ns], glu, m)
    finally:
        for name in knobs:
            qk.set_tuning(name, 0)


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
@pytest.mark.parametrize("k,n", [(6400, 17408), (6656, 5120), (6656, 11888), (7168, 11888), (8960, 11888), (9984, 4096),
                                 (16640, 5120), (19200, 1600)])
def test_slices_of_awkward_k(qk, typ, k, n):
    """Where k / 256 has few divisors a smaller image costs many slices: one token takes no more slices than
    the 32 KB image bound asks for."""
    p, bound = _plan(qk, typ, k, [n], 1), _plan(qk, typ, k, [n], 1, gemv_img_kib=32)
    assert p["kernel"] == INT8 and p["slices"] == bound["slices"]


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
def test_slices_never_jump(qk, typ):
    """Whatever k and n, one token takes at most one exchange level more than the 32 KB bound, two and four
    tokens exactly its slices."""
    for k in range(1024, 19457, 256):
        for n in (1024, 4096, 5120, 11888, 17408):
            for m in (1, 2, 4):
                p, bound = _plan(qk, typ, k, [n], m), _plan(qk, typ, k, [n], m, gemv_img_kib=32)
                if p["kernel"] != INT8:
                    continue
                assert p["slices"] in ((bound["slices"], 2 * bound["slices"]) if m == 1 else (bound["slices"],)), (k, n, m)


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
def test_slices_double_near_the_bound(qk, typ):
    """One token, k = 17408 and 5120 rows: four slices, each of whose images is half of two slices' (Q8_0 keeps
    two); 13824, where six slices would cut ranges, keeps the bound's three."""
    assert _plan(qk, typ, 17408, [5120], 1, gemv_img_kib=32)["slices"] == 2
    assert _plan(qk, typ, 17408, [5120], 1)["slices"] == (2 if typ == T_Q8_0 else 4)
    assert _plan(qk, typ, 13824, [5120], 1)["slices"] == _plan(qk, typ, 13824, [5120], 1, gemv_img_kib=32)["slices"]
    assert _plan(qk, typ, 17408, [17408], 1)["slices"] == 2  # 289 units a range


@pytest.mark.parametrize("typ,k,n,m", [(T_Q5_K, 16384, 17408, 2), (T_Q5_K, 4096, 76016, 2), (T_Q4_K, 7168, 32000, 4),
                                       (T_Q6_K, 9216, 6144, 4), (T_Q8_0, 7168, 12288, 1), (T_Q4_K, 7168, 5120, 3)])
def test_waves_kept(qk, typ, k, n, m):
    """Calls that a smaller work-group slows down run as many waves as the LDS holds."""
    p, most = _plan(qk, typ, k, [n], m), _plan(qk, typ, k, [n], m, gemv_wpg=16)
    assert p["kernel"] == INT8 and p["waves_per_group"] == most["waves_per_group"] > 8 and p["slices"] == most["slices"]


@pytest.mark.parametrize("typ,k,n,m,waves", [(T_Q4_K, 1024, 3072, 1, 8), (T_Q4_K, 5120, 17408, 1, 12), (T_Q6_K, 5120, 17408, 1, 12),
                                             (T_Q8_0, 6144, 5120, 1, 8), (T_Q4_K, 5120, 5120, 4, 12)])
def test_waves_reduced(qk, typ, k, n, m, waves):
    """Calls that run on fewer: short ranges on eight, others on a whole number per SIMD."""
    assert _plan(qk, typ, k, [n], m)["waves_per_group"] == waves < _plan(qk, typ, k, [n], m, gemv_wpg=16)["waves_per_group"]


@pytest.mark.parametrize("typ", [T_Q4_K, T_Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("m", [2, 4])
def test_min_waves_counts_what_the_lds_holds(qk, typ, m):
    """gemv_min_waves sends a call to the general kernel where the LDS holds fewer waves than it asks for, not
    where the plan takes fewer than the LDS holds."""
    k = n = 5120
    held = _plan(qk, typ, k, [n], m, gemv_wpg=16)["waves_per_group"]
    assert _plan(qk, typ, k, [n], m)["waves_per_group"] == 12 < held
    for w in (12, held):
        p = _plan(qk, typ, k, [n], m, gemv_min_waves=w)
        assert p["kernel"] == INT8 and w <= p["waves_per_group"] <= held
    if held < 16:
        assert _plan(qk, typ, k, [n], m, gemv_min_waves=held + 1)["kernel"] != INT8
