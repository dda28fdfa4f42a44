"""GPU parity of prefill calls that run as whole rounds of work-groups and a second launch over the rows
left over (one output, row stride of the whole matrix), through the C ABI: the rows at the seam and at
both ends, ragged tokens, an odd tile count at the end, the split-K sum of the second launch writing into
the wider output, and both XCD maps.  Bar as in test_gpu_gemm.py (fp16 operands, 5e-3 on both metrics).
"""
import numpy as np
import pytest

from oracle_lib import SEED_BASE, T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0, rel_errors

pytestmark = pytest.mark.gpu

TOL = 5e-3
# (type, k, n, m), sizes whose estimate favours the second launch: two and more rounds' worth of tiles
SHAPES = [(T_Q4_K, 5120, 17392, 633), (T_Q8_0, 6144, 5136, 2048), (T_Q6_K, 5120, 17408, 600), (T_Q5_K, 8192, 9232, 1010)]


@pytest.mark.parametrize("gmap", [1, 0])
@pytest.mark.parametrize("typ,k,n,m", SHAPES, ids=[f"t{t}k{k}n{n}m{m}" for t, k, n, m in SHAPES])
def test_gemm_second_launch(qk, oracle, dev, typ, k, n, m, gmap):
    w = oracle.weights(typ, n, k, SEED_BASE | 0x410)
    xh = np.random.default_rng(n + m).standard_normal((m, k), dtype=np.float32).astype(np.float16)
    W = qk.upload(w, typ, k, n, 1)
    try:
        xd, yd = dev.put(xh), dev.empty((m * n + 64) * 4)
        yd.fill_nan()
        qk.set_tuning("gemm_map", gmap)
        qk.matmul_act(W, xd.ptr, 1, m, yd.ptr, dev.stream())
        y = yd.get(np.float32, (m * n + 64,))
    finally:
        qk.set_tuning("gemm_map", 1)
        qk.free(W)
    assert np.isfinite(y[:m * n]).all() and np.isnan(y[m * n:]).all()
    y = y[:m * n].reshape(m, n)
    seams = [r for c in range(0, n, 2048) for r in (c - 1, c, c + 1) if 0 <= r < n]  # launches meet at 2048 i rows
    rows = np.unique(np.r_[0:8, seams, n - 40:n])
    toks = np.unique(np.r_[0, 31, 127, 128, m // 2, m - 2, m - 1])
    sub = w.reshape(n, -1)[rows].reshape(-1)
    ref, mag = oracle.matmul_f64(typ, sub, k, len(rows), xh[toks].astype(np.float32))
    e_max, e_norm = rel_errors(y[np.ix_(toks, rows)], ref, mag)
    assert e_max <= TOL and e_norm <= TOL, (e_max, e_norm)
