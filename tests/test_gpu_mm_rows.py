"""The row-tile matrix product (g53h_mm_f8 on FP8 matrices with 128-column blocks, replaces
src/core/glm53f_ops.c:185-228): bit-exact with the oracle at the edges of its tiles of 64 rows,
128 columns and up to two tokens, for matrices that are not 16-byte aligned, and either side of the
line to a thread per row for narrow ones."""
import ctypes as C

import numpy as np
import pytest

import glm53h
import oracle_lib as O
from glm53h import DevBuf, G53hMat, check
from test_gpu_parity import same, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return glm53h.init(0)


@pytest.mark.parametrize("rows,cols,br,T,shift", [
    (1, 5, 128, 1, 0), (64, 128, 128, 1, 0), (63, 127, 128, 2, 0), (65, 129, 16, 3, 0), (128, 136, 128, 4, 8),
    (200, 1030, 16, 5, 0), (130, 1024, 128, 9, 3), (300, 4096, 128, 2, 1), (4096, 2048, 128, 24, 0),
    (100, 1152, 128, 7, 0), (64, 2047, 64, 13, 16), (256, 2176, 128, 130, 0), (4100, 131, 128, 5, 0),
    (200, 64, 128, 3, 0), (4000, 112, 128, 4, 0), (4096, 112, 128, 5, 0), (4096, 100, 16, 24, 0), (2048, 136, 128, 24, 0),
    (2048, 207, 128, 9, 1), (2048, 208, 128, 9, 1), (2047, 180, 128, 24, 0), (2048, 135, 128, 9, 0)])
def test_mm_f8_rows(L, rows, cols, br, T, shift):
    say("mm rows", rows, cols, br, T, shift)
    rng = np.random.default_rng(rows * 7 + cols)
    w = rng.integers(0, 256, rows * cols).astype(np.uint8)
    w[(w & 0x7f) == 0x7f] ^= 1                       # no NaN codes
    sc = -(-cols // 128)
    s = rng.uniform(1e-3, 1e-1, -(-rows // br) * sc).astype(np.float32)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    wd = DevBuf.from_array(np.concatenate([np.zeros(shift, np.uint8), w]))
    sd, xd, yd = DevBuf.from_array(s), DevBuf.from_array(x), DevBuf((T * rows + 1) * 4)
    yd.upload(np.full(T * rows + 1, 7.0, np.float32))
    m = G53hMat(wd.ptr + shift, sd.ptr, rows, cols, br, 128, sc, 0)
    check(L.g53h_mm_f8(yd.ptr, xd.ptr, T, C.byref(m)), "mm")
    got = yd.download(np.float32)
    assert got[-1] == 7.0                            # nothing past the last row
    assert same(got[:-1].reshape(T, rows), O.mm_f8(O.oracle(), x, w, s, rows, cols, br, 128))


@pytest.mark.parametrize("cols,T", [(128, 262151), (16, 1048583)])
def test_mm_f8_more_outputs_than_a_grid_holds(L, cols, T):
    """So many tokens x 4096 rows that one launch has too few threads for them, by row tiles and by threads. A
    block of tokens repeated gives its result repeated, at both ends and on both sides of every multiple of
    2^16 tokens."""
    say("mm, more than a grid", cols, T)
    rows, n = 4096, 4099
    rng = np.random.default_rng(11)
    w = rng.integers(0, 256, rows * cols).astype(np.uint8)
    w[(w & 0x7f) == 0x7f] ^= 1
    s = rng.uniform(1e-3, 1e-1, rows // 128).astype(np.float32)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    wd, sd, xd, yd = DevBuf.from_array(w), DevBuf.from_array(s), DevBuf(T * cols * 4), DevBuf(T * rows * 4)
    for t in range(0, T, n):
        check(L.g53h_h2d(xd.ptr + t * cols * 4, x.ctypes.data, min(n, T - t) * cols * 4), "h2d")
    m = G53hMat(wd.ptr, sd.ptr, rows, cols, 128, 128, 1, 0)
    check(L.g53h_mm_f8(yd.ptr, xd.ptr, T, C.byref(m)), "mm")
    check(L.g53h_sync(), "sync")
    at = sorted({t for e in range(0, T, 1 << 16) for t in range(e - 2, e + 3) if t >= 0} | {T - 2, T - 1})
    want = O.mm_f8(O.oracle(), np.ascontiguousarray(x[[t % n for t in at]]), w, s, rows, cols, 128, 128)
    got = np.empty((len(at), rows), np.float32)
    for i, t in enumerate(at):
        check(L.g53h_d2h(got[i].ctypes.data, yd.ptr + t * rows * 4, rows * 4), "d2h")
    assert same(got, want)


@pytest.mark.parametrize("flags", [2, 8, 4 | 8, 4 | 16])
def test_mm_f8_refuses_tiled_codes(L, flags):
    say("mm, tiled codes", flags)
    buf = DevBuf(1 << 16)
    m = G53hMat(buf.ptr, buf.ptr, 64, 128, 1 if flags & 4 else 128, 64 if flags & 4 else 128, 2 if flags & 4 else 1, flags)
    assert L.g53h_mm_f8(buf.ptr, buf.ptr, 1, C.byref(m)) == -1
