"""Small layers (hidden up to 1024, every row of every slot at once) and small routers (scores and
selection in one launch), at the edges of their rules and over every form of descriptor that they
accept (replaces src/core/glm53f_ops.c:1144-1342). Bar: bit-exact with the oracle and with the
row-wave kernels."""
import ctypes as C

import numpy as np
import pytest

import glm53h
import glm53h.synth as S
import oracle_lib as O
from glm53h import DevBuf, G53hExpert, G53hMat, check
from test_gpu_grouped import oracle_out, run, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    return glm53h.init(0)


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("E,I,NE,K,T,kw", [
    (128, 128, 3, 1, 1, {}), (256, 128, 16, 8, 8, {}), (384, 384, 33, 8, 5, {}), (1024, 256, 64, 9, 65, {}),
    (1024, 128, 12, 4, 200, dict(shared=False)), (640, 896, 9, 8, 3, dict(norm_topk=0)),
    (256, 128, 20, 3, 70, dict(br=64)), (896, 128, 40, 16, 2, dict(limit=0.0))])
def test_small_layer_edges(L, E, I, NE, K, T, kw):
    say("small layer", E, I, NE, K, T, kw)
    sp = S.LayerSpec(E=E, I=I, NE=NE, K=K, router_sigma=0.02, **kw)
    layer = S.DeviceLayer.build(sp)
    x = S.x_host(sp, T, batch=3)
    out, idx, w = run(layer, x, 0)
    want, wi, ww = oracle_out(layer, x, idx)
    assert np.array_equal(idx, wi) and np.array_equal(bits(w), bits(ww))
    assert np.array_equal(bits(out), bits(want))


@pytest.mark.parametrize("T", [1, 7])
def test_small_layer_descriptors(L, T):
    """Octet-tiled and unaligned descriptors among row-major ones: the same values, the same result.
    Then an int4 one, as the row-wave kernels, which a layer without a block width takes."""
    say("small layer descriptors", T)
    sp = S.LayerSpec(E=384, I=256, NE=6, K=6, router_sigma=0.02)
    layer = S.DeviceLayer.build(sp)
    keep = []

    def tiled(m):
        b = DevBuf(m.rows * m.cols)
        check(L.g53h_tile_f8(b.ptr, m.w, m.rows, m.cols), "tile")
        keep.append(b)
        return G53hMat(b.ptr, m.s, m.rows, m.cols, m.br, m.bc, m.scols, 2)

    def moved(m):
        b = DevBuf(m.rows * m.cols + 16)
        check(L.g53h_d2d(b.ptr + 5, m.w, m.rows * m.cols), "d2d")
        keep.append(b)
        return G53hMat(b.ptr + 5, m.s, m.rows, m.cols, m.br, m.bc, m.scols, 0)

    def int4(m):
        q, st = DevBuf(m.rows * m.cols // 2), DevBuf(m.rows * (m.cols // 64) * 4)
        check(L.g53h_i4_from_f8(q.ptr, st.ptr, C.byref(m)), "i4")
        keep.extend((q, st))
        return G53hMat(q.ptr, st.ptr, m.rows, m.cols, 1, 64, m.cols // 64, 4)

    def put(forms):
        for e, f in forms:
            d = layer.experts[e]
            layer.experts[e] = G53hExpert(f(d.gate), f(d.up), f(d.down))
        layer.table.upload(np.frombuffer(bytes(layer.experts), np.uint8))

    x = S.x_host(sp, T, batch=4)
    want = run(layer, x, 0)
    put(((1, tiled), (2, moved), (sp.NE, tiled)))
    got = run(layer, x, 0)
    assert np.array_equal(got[1], want[1]) and np.array_equal(bits(got[0]), bits(want[0]))
    layer = S.DeviceLayer.build(sp)
    put(((3, int4),))
    got = run(layer, x, 0)
    layer.layer.block_c = 0
    want = run(layer, x, 0)
    assert np.array_equal(got[1], want[1]) and np.array_equal(bits(got[0]), bits(want[0]))


@pytest.mark.parametrize("block_c", [128, 0])
@pytest.mark.parametrize("flags", [8, 4 | 8, 4 | 16])
def test_unreadable_layouts_give_nan(L, flags, block_c):
    """A descriptor in a layout that the small-layer and row kernels do not read (MFMA-tiled, int4-tiled):
    NaN for the tokens that chose the expert, not a misread one; the other tokens as before."""
    say("small layer, unreadable layout", flags, block_c)
    sp = S.LayerSpec(E=384, I=256, NE=8, K=2, router_sigma=0.05)
    layer = S.DeviceLayer.build(sp)
    layer.layer.block_c = block_c
    x = S.x_host(sp, 9, batch=8)
    want, idx, _ = run(layer, x, 0)
    d = layer.experts[3]
    layer.experts[3] = G53hExpert(*[G53hMat(m.w, m.s, m.rows, m.cols, 1 if flags & 4 else m.br, 64 if flags & 4 else m.bc,
                                            m.cols // (64 if flags & 4 else 128), flags) for m in (d.gate, d.up, d.down)])
    layer.table.upload(np.frombuffer(bytes(layer.experts), np.uint8))
    got, idx1, _ = run(layer, x, 0)
    assert np.array_equal(idx, idx1)
    hit = (idx == 3).any(axis=1)
    assert hit.any() and not hit.all()
    assert np.isnan(got[hit]).all() and np.array_equal(bits(got[~hit]), bits(want[~hit]))


@pytest.mark.parametrize("T,NE,E,K,shift", [
    (1, 1, 128, 1, 0), (1, 32, 256, 8, 0), (2, 65, 384, 8, 0), (3, 16, 4096, 16, 0), (512, 128, 512, 4, 0),
    (200, 320, 128, 10, 0), (512, 129, 128, 3, 0), (5, 33, 256, 8, 1),
    (257, 64, 256, 8, 0), (64, 321, 2048, 8, 0), (33, 1024, 1024, 8, 0), (17, 129, 768, 8, 0), (700, 300, 2048, 8, 0), (2000, 288, 512, 8, 0),
    (4100, 30, 2048, 8, 0), (16400, 100, 512, 4, 0)])
def test_small_router(L, T, NE, E, K, shift):
    """Either side of the rule, and the matrix-core form over one and several column ranges of one and
    more chunks, in either order of its tiles; shift moves x off 16-byte alignment."""
    say("small router", T, NE, E, K, shift)
    sp = S.LayerSpec(E=E, I=128, NE=NE, K=K, router_sigma=0.05)
    rf, bias = S.router_host(sp), S.bias_host(sp)
    x = S.x_host(sp, T, batch=5)
    xd = DevBuf(x.nbytes + 16)
    check(L.g53h_h2d(xd.ptr + 4 * shift, x.ctypes.data, x.nbytes), "h2d")
    g, b = DevBuf.from_array((rf.view(np.uint32) >> 16).astype(np.uint16)), DevBuf.from_array(bias)
    idx, w, flag = DevBuf(T * K * 4), DevBuf(T * K * 4), DevBuf(4)
    flag.zero()
    check(L.g53h_router(idx.ptr, w.ptr, xd.ptr + 4 * shift, T, g.ptr, 1, b.ptr, NE, E, K, sp.norm_topk,
                        C.c_float(sp.routed_scale), flag.ptr), "router")
    wi, ww = O.router(O.oracle(), x, sp, rf, bias)
    assert np.array_equal(idx.download(np.int32).reshape(T, K), wi)
    assert np.array_equal(bits(w.download(np.float32).reshape(T, K)), bits(ww))
    assert flag.download(np.int32)[0] == 0


def test_router_more_tokens_than_grid_rows(L):
    """1,048,592 tokens, 65,537 tiles of 16: a block of tokens repeated gives its result repeated."""
    say("router, a million tokens")
    E, NE, K, n, reps = 256, 20, 4, 4096, 256
    T = n * reps + 16
    sp = S.LayerSpec(E=E, I=128, NE=NE, K=K, router_sigma=0.05)
    rf, bias = S.router_host(sp), S.bias_host(sp)
    x = S.x_host(sp, n, batch=7)
    xd = DevBuf(T * E * 4)
    check(L.g53h_h2d(xd.ptr, x.ctypes.data, x.nbytes), "h2d")
    have = n
    while have < T:                                  # doubling copies
        m = min(have, T - have)
        check(L.g53h_d2d(xd.ptr + have * E * 4, xd.ptr, m * E * 4), "d2d")
        have += m
    g, b = DevBuf.from_array((rf.view(np.uint32) >> 16).astype(np.uint16)), DevBuf.from_array(bias)
    idx, w = DevBuf(T * K * 4), DevBuf(T * K * 4)
    check(L.g53h_router(idx.ptr, w.ptr, xd.ptr, T, g.ptr, 1, b.ptr, NE, E, K, sp.norm_topk,
                        C.c_float(sp.routed_scale), None), "router")
    wi, ww = O.router(O.oracle(), x, sp, rf, bias)
    at = np.arange(T) % n
    assert np.array_equal(idx.download(np.int32).reshape(T, K), wi[at])
    assert np.array_equal(bits(w.download(np.float32).reshape(T, K)), bits(ww)[at])


def test_small_router_nan(L):
    """A token whose scores are NaN raises the flag, the others are as without it."""
    say("small router NaN")
    sp = S.LayerSpec(E=256, I=128, NE=16, K=4, router_sigma=0.05)
    layer = S.DeviceLayer.build(sp)
    x = S.x_host(sp, 3, batch=6)
    xn = x.copy()
    xn[1, 17] = np.nan
    res = []
    for v in (x, xn):
        xd = DevBuf.from_array(v)
        idx, w, flag = DevBuf(3 * 4 * 4), DevBuf(3 * 4 * 4), DevBuf(4)
        flag.zero()
        check(L.g53h_router(idx.ptr, w.ptr, xd.ptr, 3, layer.router.ptr, 1, layer.bias.ptr, 16, 256, 4, 1,
                            C.c_float(2.5), flag.ptr), "router")
        res.append((idx.download(np.int32).reshape(3, 4), bits(w.download(np.float32).reshape(3, 4)),
                    flag.download(np.int32)[0]))
    assert res[0][2] == 0 and res[1][2] != 0
    for t in (0, 2):
        assert np.array_equal(res[0][0][t], res[1][0][t]) and np.array_equal(res[0][1][t], res[1][1][t])
