"""The grouped GEMMs' step pipeline at the edges of its tiles (32 and 64 positions), of its shortest
and longest items (4 to 32 steps), over both code layouts and over codes that are not 16-byte
aligned (replaces src/core/glm53f_ops.c:376-444 in :1144-1342). Every expert is chosen by every
token, so a tile's positions are the batch's tokens. Bar: routing bit-exact, outputs within the
path's tolerance of the oracle."""
import ctypes as C

import numpy as np
import pytest

import glm53h
import glm53h.synth as S
from glm53h import DevBuf, G53hExpert, G53hMat, check
from test_gpu_grouped import oracle_out, run, say, within

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return glm53h.init(0)


@pytest.mark.parametrize("E,inter,T,tiled", [
    (512, 512, 2, True), (512, 512, 32, False), (512, 1024, 33, True), (1024, 512, 64, False),
    (1024, 1024, 65, True), (2048, 512, 97, False), (512, 2048, 129, True), (4096, 512, 31, True),
    (512, 4096, 63, False)])
def test_grouped_tile_edges(L, E, inter, T, tiled):
    say("tile edges", E, inter, T, tiled)
    sp = S.LayerSpec(E=E, I=inter, NE=3, K=3, router_sigma=0.02)
    layer = S.DeviceLayer.build(sp, tiled=tiled)
    x = S.x_host(sp, T, batch=1)
    out, idx, w = run(layer, x, 1, "g53h_moe_grouped")
    want, wi, ww = oracle_out(layer, x, idx)
    assert np.array_equal(idx, wi) and np.array_equal(w.view(np.uint32), ww.view(np.uint32))
    within(out, want, f"E={E} I={inter} T={T}")


@pytest.mark.parametrize("shift,T,tiled", [(1, 5, False), (4, 40, True), (8, 130, False)])
def test_grouped_unaligned_codes(L, shift, T, tiled):
    """The second expert's codes at an address that is not a multiple of 16, the others aligned: the
    result is bit for bit that of the aligned layer."""
    say("unaligned codes", shift, T, tiled)
    sp = S.LayerSpec(E=1024, I=512, NE=4, K=3, router_sigma=0.02)
    layer = S.DeviceLayer.build(sp, tiled=tiled)
    x = S.x_host(sp, T, batch=2)
    want, wi, _ = run(layer, x, 1, "g53h_moe_grouped")
    keep = []

    def moved(m):
        b = DevBuf(m.rows * m.cols + 16)
        check(L.g53h_d2d(b.ptr + shift, m.w, m.rows * m.cols), "d2d")
        keep.append(b)
        return G53hMat(b.ptr + shift, m.s, m.rows, m.cols, m.br, m.bc, m.scols, m.flags)

    e = layer.experts[1]
    layer.experts[1] = G53hExpert(moved(e.gate), moved(e.up), moved(e.down))
    layer.table.upload(np.frombuffer(bytes(layer.experts), np.uint8))
    out, idx, _ = run(layer, x, 1, "g53h_moe_grouped")
    assert np.array_equal(idx, wi)
    assert np.array_equal(out.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("E,inter,T", [(512, 512, 2), (512, 4096, 33), (4096, 512, 65), (1024, 2048, 130), (2048, 1024, 5)])
def test_grouped_mfma_tiled(L, E, inter, T):
    """MFMA-tiled experts (the drop-in's cache may hold them), whose addresses depend on both sizes: bit for
    bit the row-major layer."""
    say("grouped, MFMA-tiled", E, inter, T)
    sp = S.LayerSpec(E=E, I=inter, NE=4, K=3, router_sigma=0.02)
    x = S.x_host(sp, T, batch=5)
    want, wi, ww = run(S.DeviceLayer.build(sp), x, 1, "g53h_moe_grouped")
    layer = S.DeviceLayer.build(sp, mfma=True)
    begin = L.g53h_grouped_begin_layout
    begin.argtypes, begin.restype = [C.c_void_p, C.c_int, C.POINTER(glm53h.G53hMoeLayer), C.c_void_p, C.c_int], C.c_int
    xd, od, id_, wd = DevBuf.from_array(x), DevBuf(x.nbytes), DevBuf.from_array(wi), DevBuf.from_array(ww)
    check(begin(xd.ptr, T, C.byref(layer.layer), id_.ptr, 2), "begin")
    check(L.g53h_grouped_batch(C.byref(layer.layer)), "batch")
    check(L.g53h_grouped_end(od.ptr, wd.ptr), "end")
    assert L.g53h_grouped_errors() == 0
    assert np.array_equal(od.download(np.uint32).reshape(x.shape), want.view(np.uint32))


def test_trace_stays_in_its_buffer(L):
    """g53h_set_grouped_trace writes 8 words for each gate/up item and nothing after them."""
    say("grouped trace")
    sp = S.LayerSpec(E=512, I=512, NE=3, K=3, router_sigma=0.02)
    layer = S.DeviceLayer.build(sp)
    items = (sp.NE + 1) * sp.I // 128                # five tokens: a tile of each expert and the shared one
    buf = DevBuf(items * 32 * 8)
    buf.zero()
    check(L.g53h_set_grouped_trace(buf.ptr), "trace")
    try:
        run(layer, S.x_host(sp, 5, batch=3), 1, "g53h_moe_grouped")
    finally:
        check(L.g53h_set_grouped_trace(None), "trace")
    got = buf.download(np.uint64)
    t = got[:items * 8].reshape(items, 8)
    assert (t[:, 0] > 0).all() and (t[:, 2] >= t[:, 0]).all() and (t[:, 3] >= t[:, 2]).all()
    assert not got[items * 8:].any()


@pytest.mark.parametrize("tiled,flags", [(False, 8), (True, 8), (True, 2 | 8), (False, 16), (False, 2), (True, 0)])
def test_grouped_other_layouts_are_unusable(L, tiled, flags):
    """A descriptor marked with any layout but the pass's: flag 8, and the expert's share is zero, as that of
    a layer without it."""
    say("grouped, other layout", tiled, flags)
    sp = S.LayerSpec(E=512, I=512, NE=3, K=3, router_sigma=0.02)
    x = S.x_host(sp, 5, batch=4)
    outs = []
    for missing in (False, True):
        layer = S.DeviceLayer.build(sp, tiled=tiled)
        e = layer.experts[1]
        layer.experts[1] = G53hExpert() if missing else G53hExpert(
            *[G53hMat(m.w, m.s, m.rows, m.cols, m.br, m.bc, m.scols, flags) for m in (e.gate, e.up, e.down)])
        layer.table.upload(np.frombuffer(bytes(layer.experts), np.uint8))
        L.g53h_grouped_errors()
        xd, od = DevBuf.from_array(x), DevBuf(x.nbytes)
        check(L.g53h_moe_grouped(od.ptr, xd.ptr, 5, C.byref(layer.layer), None, None), "grouped")
        assert L.g53h_grouped_errors() == (0 if missing else 8)
        outs.append(od.download(np.uint32))
    assert np.array_equal(*outs)
