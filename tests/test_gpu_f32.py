"""GPU checks of the F32-weight kernels at the edges of their forms, through the C ABI: every token count
around a pass (1, 4, 8, 16), row counts that leave rows of a work-group or a tile empty, k with one and
with an odd number of 256-element runs, large calls on MFMA tiles, and groups whose F32 matrices of
different heights share a launch.

Bar: a sum is a chain of at most k / 256 fp32 FMAs per lane (k / 512 * 8 per tile slot) and under 20
further additions, each within 2^-24 of its running magnitude: below 2e-6 of sum|w x| at k = 5120.
"""
import numpy as np
import pytest

from oracle_lib import SEED_BASE, rel_errors

pytestmark = pytest.mark.gpu

T_F32 = 0
TOL = 2e-6
F32, F16, F16X = 0, 1, 2


def _xperm(a):
    i = np.arange(a.shape[1])
    out = np.empty_like(a)
    out[:, (i & ~1023) | (((i >> 3) & 3) << 8) | (((i >> 8) & 3) << 6) | (((i >> 5) & 7) << 3) | (i & 7)] = a
    return out


def _weights(n, k, seed):
    return np.random.default_rng(seed).standard_normal((n, k)).astype(np.float32).view(np.uint8).reshape(-1)


# (k, n, m): rows 1 / 2 / 4 per work-group, four, eight and sixteen tokens a pass, MFMA tiles
SHAPES = [(256, 1, 1), (1280, 3, 2), (5120, 48, 4), (768, 5, 5), (256, 17, 9), (5120, 48, 13), (1024, 130, 17),
          (1280, 127, 22), (256, 1031, 8), (1024, 2050, 15), (256, 4099, 6), (8448, 1030, 13), (256, 97, 1025),
          (1280, 1601, 63), (768, 33, 3001),
          # a wave per two or four rows (k <= 768, many rows), ragged rows and tokens, one past its longest k
          (256, 4097, 1), (512, 5003, 3), (768, 1027, 16), (256, 2052, 7), (512, 1500, 11), (768, 4099, 1), (1024, 4099, 1),
          # 16 x 16 tiles: at 256 tiles and one past, ragged rows and tokens, on the line of 44 Ki outputs
          (1280, 4096, 11), (256, 4091, 16), (768, 4097, 13), (2304, 44, 1024), (256, 47, 1013), (5120, 241, 255),
          # the same on xperm x
          (1024, 4096, 11), (2048, 3009, 15)]


@pytest.mark.parametrize("k,n,m", SHAPES, ids=[f"k{k}n{n}m{m}" for k, n, m in SHAPES])
def test_f32_edges(qk, oracle, dev, k, n, m):
    w = _weights(n, k, n + m)
    xh = oracle.normal(SEED_BASE | (0x300 + m), m * k).reshape(m, k).astype(np.float16)
    wd, outs = dev.put(w), []
    W = qk.weight_view(wd.ptr, T_F32, k, n, 0)
    fmts = [(F32, xh.astype(np.float32)), (F16, xh)] + ([(F16X, _xperm(xh))] if m < 16 and k % 1024 == 0 else [])
    for fmt, xa in fmts:
        xd, yd = dev.put(xa), dev.empty((m * n + 64) * 4)
        yd.fill_nan()
        qk.matmul_act(W, xd.ptr, fmt, m, yd.ptr, dev.stream())
        y = yd.get(np.float32, (m * n + 64,))
        assert np.isnan(y[m * n:]).all()  # nothing past the last row of the last token
        outs.append(y[:m * n].reshape(m, n))
    toks = np.unique(np.r_[0:min(m, 40), max(0, m - 40):m])
    ref, mag = oracle.matmul_f64(T_F32, w, k, n, xh[toks].astype(np.float32))
    for y in outs:
        assert np.array_equal(y.view(np.uint32), outs[0].view(np.uint32))  # fp16 widens exactly
        e_max, e_norm = rel_errors(y[toks], ref, mag)
        assert np.isfinite(y).all() and e_max < TOL and e_norm < TOL, (e_max, e_norm)


@pytest.mark.parametrize("m", [1, 3, 13])
def test_f32_group_heights(qk, oracle, dev, m):
    """F32 matrices of different heights in one group: each output is what the matrix gives alone."""
    k, ns = 1024, (48, 7, 130, 1)
    ws = [_weights(n, k, 40 + n) for n in ns]
    x = oracle.normal(SEED_BASE | (0x340 + m), m * k).reshape(m, k)
    bufs, xd = [dev.put(w) for w in ws], dev.put(x)
    Ws = [qk.weight_view(b.ptr, T_F32, k, n, 0) for b, n in zip(bufs, ns)]
    ys = [dev.empty(m * n * 4) for n in ns]
    for y in ys:
        y.fill_nan()
    qk.gemv_group(Ws, [y.ptr for y in ys], False, xd.ptr, m, dev.stream())
    for w, n, y in zip(ws, ns, ys):
        ref, mag = oracle.matmul_f64(T_F32, w, k, n, x)
        e_max, e_norm = rel_errors(y.get(np.float32, (m, n)), ref, mag)
        assert e_max < TOL and e_norm < TOL, (n, e_max, e_norm)


@pytest.mark.parametrize("n,m", [(128, 800), (100, 1001), (48, 960), (3000, 17)])
def test_f32_tile_sums(qk, dev, n, m):
    """MFMA tiles sum as closely as the row kernels.  With u = 2.5e-8 the root mean square of an fp32 rounding, k
    = 5120 random-sign products in passes of 32, 10 passes a wave and 16 waves give sqrt(16 + 5.5 + 8.5) u =
    1.4e-7 of the result's 2-norm (one chain of 320 a wave: sqrt(160 + 8.5) u = 3.2e-7).
    """
    k = 5120
    w = _weights(n, k, n + m)
    xh = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
    wd, xd, yd = dev.put(w), dev.put(xh), dev.empty(m * n * 4)
    qk.matmul_act(qk.weight_view(wd.ptr, T_F32, k, n, 0), xd.ptr, F16, m, yd.ptr, dev.stream())
    ref = xh.astype(np.float64) @ w.view(np.float32).reshape(n, k).astype(np.float64).T
    err = np.linalg.norm(yd.get(np.float32, (m, n)) - ref) / np.linalg.norm(ref)
    assert err < 1.9e-7, err


def test_f32_group_on_tiles(qk, oracle, dev):
    """A group of 44 Ki outputs and more: matrices of different heights on 16 x 16 tiles, one per grid z."""
    k, m, ns = 1024, 13, (2048, 1031, 512, 7)
    assert sum(ns) * m >= 44 * 1024 and sum(-(-n // 16) for n in ns) <= 256
    ws = [_weights(n, k, 60 + n) for n in ns]
    xh = oracle.normal(SEED_BASE | 0x350, m * k).reshape(m, k).astype(np.float16)
    bufs = [dev.put(w) for w in ws]
    Ws = [qk.weight_view(b.ptr, T_F32, k, n, 0) for b, n in zip(bufs, ns)]
    for fmt, xa in ((F32, xh.astype(np.float32)), (F16, xh), (F16X, _xperm(xh))):
        xd, ys = dev.put(xa), [dev.empty((m * n + 64) * 4) for n in ns]
        for y in ys:
            y.fill_nan()
        qk.gemv_group_act(Ws, [y.ptr for y in ys], False, xd.ptr, fmt, m, F32, dev.stream())
        for w, n, yd in zip(ws, ns, ys):
            y = yd.get(np.float32, (m * n + 64,))
            assert np.isnan(y[m * n:]).all()
            ref, mag = oracle.matmul_f64(T_F32, w, k, n, xh.astype(np.float32))
            e_max, e_norm = rel_errors(y[:m * n].reshape(m, n), ref, mag)
            assert e_max < TOL and e_norm < TOL, (n, fmt, e_max, e_norm)
