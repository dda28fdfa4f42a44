"""GPU checks of the GEMM's launches of several matrices, which few-token calls take only where the few-token kernel
has no plan or a knob asks for a plan of the GEMM: groups (a matrix per grid z, split-K sums of different
heights) and gate/up pairs (k_glu_sum), under forced K-parts and tile pairs, and a k whose x slices the few-token
kernel's LDS does not hold.  Bar: fp16 operands (5e-3 on both metrics, x rounded for the reference).
"""
import numpy as np
import pytest

from oracle_lib import SEED_BASE, T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0, rel_errors
from test_few_plan import _plan as few_plan

pytestmark = pytest.mark.gpu

TYPES = [T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0]
IDS = ["q4k", "q5k", "q6k", "q8_0"]
TOL = 5e-3
KNOBS = [("gemm_ksplit", 1), ("gemm_ksplit", 3), ("gemm_pairs", 4), ("gemm_pairs", 8)]


def _run(qk, oracle, dev, typ, k, ns, m, glu, knob=None):
    ws = [oracle.weights(typ, n, k, SEED_BASE | (0x420 + i)) for i, n in enumerate(ns)]
    xh = oracle.normal(SEED_BASE | (0x430 + m), m * k).reshape(m, k).astype(np.float16)
    Ws = [qk.upload(w, typ, k, n, 1) for w, n in zip(ws, ns)]
    outs = ns[:1] if glu else ns
    try:
        xd, ys = dev.put(xh), [dev.empty((m * n + 64) * 4) for n in outs]
        for y in ys:
            y.fill_nan()
        if knob:
            qk.set_tuning(*knob)
        qk.gemv_group_act(Ws, [y.ptr for y in ys], glu, xd.ptr, 1, m, 0, dev.stream())
        got = [y.get(np.float32, (m * n + 64,)) for y, n in zip(ys, outs)]
    finally:
        if knob:
            qk.set_tuning(knob[0], 0)
        for W in Ws:
            qk.free(W)
    refs = [oracle.matmul_f64(typ, w, k, n, xh.astype(np.float32)) for w, n in zip(ws, ns)]
    for y, n in zip(got, outs):
        assert np.isfinite(y[:m * n]).all() and np.isnan(y[m * n:]).all()
    got = [y[:m * n].reshape(m, n) for y, n in zip(got, outs)]
    if glu:
        g, u = refs[0][0], refs[1][0]
        ref = g / (1.0 + np.exp(-g)) * u
        assert np.linalg.norm(got[0] - ref) / np.linalg.norm(ref) < TOL
        assert np.abs(got[0] - ref).max() <= TOL * np.abs(ref).max()
        return
    for y, (ref, mag) in zip(got, refs):
        e_max, e_norm = rel_errors(y, ref, mag)
        assert e_max <= TOL and e_norm <= TOL, (e_max, e_norm)


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
@pytest.mark.parametrize("knob", KNOBS, ids=[f"{n}{v}" for n, v in KNOBS])
@pytest.mark.parametrize("m", [5, 13])
def test_group(qk, oracle, dev, typ, knob, m):
    _run(qk, oracle, dev, typ, 2048, (1040, 16, 48, 336), m, False, knob)


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
@pytest.mark.parametrize("knob", KNOBS, ids=[f"{n}{v}" for n, v in KNOBS])
@pytest.mark.parametrize("k,n,m", [(2304, 336, 8), (1024, 80, 15)])
def test_pair(qk, oracle, dev, typ, knob, k, n, m):
    _run(qk, oracle, dev, typ, k, (n, n), m, True, knob)


@pytest.mark.parametrize("typ", [T_Q4_K, T_Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("ns,glu", [((48,), False), ((48, 16), False), ((48, 48), True)], ids=["one", "group", "pair"])
def test_no_few_token_plan(qk, oracle, dev, typ, ns, glu):
    k, m = 131072, 13
    assert few_plan(qk, typ, k, list(ns), m, pair=glu)[0] is None
    _run(qk, oracle, dev, typ, k, ns, m, glu)
