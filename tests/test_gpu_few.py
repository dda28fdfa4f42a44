"""GPU checks of the few-token GEMM (5..16 tokens) at the edges of its plan, through the C ABI: one
super-block, K-slices of unequal length, fewer units than waves, tiles cut between two and more waves, a
tile count that leaves work-groups unequal, eight and sixteen token slots with and without padding, the
xperm layout (bitwise equal to plain), and matrices of different heights in one launch.

Bar: the operands are rounded to fp16 as in the GEMM (5e-3 on both metrics, x rounded for the reference).
"""
import numpy as np
import pytest

from oracle_lib import SEED_BASE, T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0, rel_errors
from test_few_plan import _plan

pytestmark = pytest.mark.gpu

TYPES = [T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0]
IDS = ["q4k", "q5k", "q6k", "q8_0"]
F16, F16X = 1, 2
TOL = 5e-3


def _xperm(a):
    i = np.arange(a.shape[1])
    out = np.empty_like(a)
    out[:, (i & ~1023) | (((i >> 3) & 3) << 8) | (((i >> 8) & 3) << 6) | (((i >> 5) & 7) << 3) | (i & 7)] = a
    return out


SHAPES = [(256, 16, 5), (768, 48, 16), (1024, 2064, 8), (2304, 208, 9), (3072, 5120, 13), (7168, 336, 15),
          (17408, 272, 6), (1024, 17408, 16)]


@pytest.mark.parametrize("typ", TYPES, ids=IDS)
@pytest.mark.parametrize("k,n,m", SHAPES, ids=[f"k{k}n{n}m{m}" for k, n, m in SHAPES])
def test_few_edges(qk, oracle, dev, typ, k, n, m):
    w = oracle.weights(typ, n, k, SEED_BASE | (0x3A0 + m))
    xh = oracle.normal(SEED_BASE | (0x3C0 + m), m * k).reshape(m, k).astype(np.float16)
    W = qk.upload(w, typ, k, n, 1)
    ys = []
    try:
        for fmt, xa in [(F16, xh)] + ([(F16X, _xperm(xh))] if k % 1024 == 0 and m < 16 else []):
            xd, yd = dev.put(xa), dev.empty((m * n + 64) * 4)
            yd.fill_nan()
            for _ in range(2):  # a second call finds nothing left behind by the first
                qk.matmul_act(W, xd.ptr, fmt, m, yd.ptr, dev.stream())
            y = yd.get(np.float32, (m * n + 64,))
            assert np.isnan(y[m * n:]).all()
            ys.append(y[:m * n].reshape(m, n))
    finally:
        qk.free(W)
    rows = np.unique(np.r_[0:min(n, 80), max(0, n - 80):n])
    sub = w.reshape(n, -1)[rows].reshape(-1)
    ref, mag = oracle.matmul_f64(typ, sub, k, len(rows), xh.astype(np.float32))
    for y in ys:
        assert np.isfinite(y).all()
        assert np.array_equal(y.view(np.uint32), ys[0].view(np.uint32))
        e_max, e_norm = rel_errors(y[:, rows], ref, mag)
        assert e_max <= TOL and e_norm <= TOL, (e_max, e_norm)


@pytest.mark.parametrize("m", [5, 8, 13])
def test_few_group_heights(qk, oracle, dev, m):
    """Four matrices of different heights in one launch: each is what it gives alone, bitwise only where
    the plan is the same, so against the oracle."""
    k, ns = 2048, (1040, 16, 48, 336)
    ws = [oracle.weights(T_Q4_K, n, k, SEED_BASE | (0x3E0 + i)) for i, n in enumerate(ns)]
    xh = oracle.normal(SEED_BASE | (0x3F0 + m), m * k).reshape(m, k).astype(np.float16)
    Ws = [qk.upload(w, T_Q4_K, k, n, 1) for w, n in zip(ws, ns)]
    try:
        xd, ys = dev.put(xh), [dev.empty(m * n * 4) for n in ns]
        for y in ys:
            y.fill_nan()
        qk.gemv_group_act(Ws, [y.ptr for y in ys], False, xd.ptr, F16, m)
        outs = [y.get(np.float32, (m, n)) for y, n in zip(ys, ns)]
    finally:
        for W in Ws:
            qk.free(W)
    for w, n, y in zip(ws, ns, outs):
        ref, mag = oracle.matmul_f64(T_Q4_K, w, k, n, xh.astype(np.float32))
        e_max, e_norm = rel_errors(y, ref, mag)
        assert e_max <= TOL and e_norm <= TOL, (n, e_max, e_norm)


# (type, k, n, m, waves): 128 units and more a work-group, so twelve waves, rings refilled many times and tiles cut
# between the waves; Q8_0 whose LDS holds eight
TALL = [(t, 1024, 131088, m, 12) for t in TYPES for m in (8, 13)] + [(T_Q8_0, 4096, 28704, 8, 8)]


@pytest.mark.parametrize("typ,k,n,m,waves", TALL, ids=[f"{IDS[TYPES.index(t)]}k{k}m{m}" for t, k, n, m, _ in TALL])
def test_few_many_units(qk, oracle, dev, typ, k, n, m, waves):
    """Every row of a tall matrix whose rows repeat every 1040 (65 tiles, no multiple of a work-group's)."""
    plan, _ = _plan(qk, typ, k, [n], m)
    units = -(-plan.ntiles // plan.wgs) * -(-plan.nsb // plan.slices)
    assert plan.waves == waves and units >= 128
    base = 1040
    w = oracle.weights(typ, base, k, SEED_BASE | (0x440 + m)).reshape(base, -1)
    xh = oracle.normal(SEED_BASE | (0x450 + m), m * k).reshape(m, k).astype(np.float16)
    W = qk.upload(np.ascontiguousarray(np.resize(w, (n, w.shape[1]))).reshape(-1), typ, k, n, 1)
    ys = []
    try:
        for fmt, xa in ((F16, xh), (F16X, _xperm(xh))):
            xd, yd = dev.put(xa), dev.empty((m * n + 64) * 4)
            yd.fill_nan()
            qk.matmul_act(W, xd.ptr, fmt, m, yd.ptr, dev.stream())
            y = yd.get(np.float32, (m * n + 64,))
            assert np.isfinite(y[:m * n]).all() and np.isnan(y[m * n:]).all()
            ys.append(y[:m * n].reshape(m, n))
    finally:
        qk.free(W)
    assert np.array_equal(ys[0].view(np.uint32), ys[1].view(np.uint32))
    ref, mag = oracle.matmul_f64(typ, w.reshape(-1), k, base, xh.astype(np.float32))
    rows = np.arange(n) % base
    e_max, e_norm = rel_errors(ys[0], ref[:, rows], mag[:, rows])
    assert e_max <= TOL and e_norm <= TOL, (e_max, e_norm)
