"""GPU checks of the layout change at the edges of its chunks, through the C ABI: one super-block, chunk
counts that do not divide, row starts at every even offset of a 16-byte word (Q6_K), one and many tiles.
The T16 bytes are read back through the bit-exact row dequant (whose byte maps tests/test_layout.py
checks), the way back must restore the file's bytes, and neither may touch what follows the tensor.
"""
import numpy as np
import pytest

from oracle_lib import SEED_BASE, T_Q4_K, T_Q5_K, T_Q6_K, T_Q8_0

pytestmark = pytest.mark.gpu

SHAPES = [(256, 16), (512, 48), (2048, 32), (2304, 16), (4352, 80), (5120, 272), (17408, 16), (7936, 400),
          # chunks of two, four and eight super-blocks (the shapes above: one)
          (4352, 1360), (7936, 1600), (5888, 6400)]
GUARD = 256


@pytest.mark.parametrize("typ", [T_Q8_0, T_Q4_K, T_Q5_K, T_Q6_K], ids=["q8_0", "q4k", "q5k", "q6k"])
@pytest.mark.parametrize("k,n", SHAPES, ids=[f"k{k}n{n}" for k, n in SHAPES])
def test_repack_edges(qk, oracle, dev, typ, k, n):
    w = oracle.weights(typ, n, k, SEED_BASE | (0x380 + n))
    src, mark = dev.put(w), np.full(w.size + GUARD, 0xA5, np.uint8)
    t16, back = dev.put(mark), dev.put(mark)
    G = qk.weight_view(src.ptr, typ, k, n, 0)
    T = qk.repack(G, t16.ptr, 1)
    qk.repack(T, back.ptr, 0)
    a, b = t16.get(np.uint8, (mark.size,)), back.get(np.uint8, (mark.size,))
    assert np.array_equal(b[:w.size], w)
    assert (a[w.size:] == 0xA5).all() and (b[w.size:] == 0xA5).all()
    rows = np.unique(np.r_[0:min(n, 33), max(0, n - 17):n]).astype(np.int32)
    rd, out = dev.put(rows), dev.empty(len(rows) * k * 4)
    qk.dequant_rows(T, rd.ptr, len(rows), out.ptr)
    got = out.get(np.float32, (len(rows), k))
    assert np.array_equal(got.view(np.uint32), oracle.dequant_matrix(typ, w, k, n)[rows].view(np.uint32))
