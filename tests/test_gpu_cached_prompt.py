"""Several tokens through the HBM cache (glm53f_moe, T >= 2; src/core/glm53f_ops.c:1144-1362): a cache
with slots for every expert a pass may name is multiplied in one grouped pass, a smaller one chunk by
chunk and batch by batch. Both make the reference's calls, so the outputs are equal bit for bit, as are
the counts of gets, with octet-tiled and MFMA-tiled slots, hints on and off, and a get that fails."""
import ctypes as C

import numpy as np
import pytest

import glm53h
import glm53h.synth as S
import oracle_lib as O
from glm53h import check
from test_gpu_cache import make_cfg
from test_gpu_grouped import within
from test_gpu_i4 import dev_quant, imat
from test_gpu_parity import fmat, say

pytestmark = pytest.mark.gpu
NP = 6


@pytest.fixture(scope="module")
def L():
    return glm53h.init(0)


@pytest.fixture(scope="module")
def layer():
    sp = S.spec(2, NE=24, seed=5)
    pool = [S.expert_host(sp, p) for p in range(NP)]
    return sp, pool, S.router_host(sp), S.bias_host(sp), S.expert_host(sp, "shared")


def run(L, layer, x, slots, n_io=0, prefetch_n=0, fails=(), shared=True, hold=None, reads=None,
        predict=False):
    sp, pool, W, B, sh = layer
    cf = make_cfg(sp)
    cf.n_layers = 1

    def view(_st, _layer, e, out):
        if e in fails:
            return -1
        if reads is not None:                        # started and not handed back yet
            reads.append(e)
            most[0] = max(most[0], len(reads))
        q = out.contents
        q.gate, q.up, q.down = [fmat(w, s, r, c, 128, 128) for (w, s), (r, c) in
                                zip(pool[e % NP], [(sp.I, sp.E), (sp.I, sp.E), (sp.E, sp.I)])]
        return 0

    most = [0]
    back = glm53h.DONE_FN(lambda _st, _layer, e: reads.remove(e)) if reads is not None else glm53h.DONE_FN()
    st = glm53h.G53hStore(glm53h.VIEW_FN(view), back, None)
    c, probe = glm53h.Glm53fCache(), glm53h.Glm53fCache()
    check(L.g53h_cache_init_store(C.byref(probe), C.byref(st), C.byref(cf), 1 << 30, 0, 0), "cache")
    most[0] = 0
    budget = probe.slot_bytes * slots
    L.glm53f_cache_free(C.byref(probe))
    check(L.g53h_cache_init_store(C.byref(c), C.byref(st), C.byref(cf), budget, n_io, 0), "cache")
    w = glm53h.Glm53fMoeW()
    w.gate, w.bias, w.src, w.prefetch_n = W.ctypes.data, B.ctypes.data, C.pointer(c.src), prefetch_n
    w.sh_gate, w.sh_up, w.sh_down = [m if isinstance(m, glm53h.Glm53fMat) else fmat(*m, r, c, 128, 128) for m, (r, c) in
                                     zip(sh, [(sp.I, sp.E), (sp.I, sp.E), (sp.E, sp.I)])]
    if predict:
        w.next_gate, w.next_bias, w.prefill_next = W.ctypes.data, B.ctypes.data, 1
    drops = C.c_long.in_dll(L, "glm53f_expert_drops")
    was, outs = drops.value, []
    done = hold(c) if hold else None
    try:
        for _ in range(2):                           # the second call finds what fits resident
            out = np.zeros(x.shape, np.float32)
            (L.glm53f_moe if shared else L.glm53f_moe_routed)(out.ctypes.data, x.ctypes.data, C.byref(w), C.byref(cf),
                                                              x.shape[0], None)
            outs.append(out)
        if done:
            done()
        check(L.glm53f_cache_sync(C.byref(c)), "sync")
        gets, pins = c.hits + c.misses, sum(c.pins[i] for i in range(c.nslot))
    finally:
        L.glm53f_cache_free(C.byref(c))
        L.glm53f_forget_host_weights()
    assert pins == 0                                 # everything was released
    lost, drops.value = drops.value - was, was
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    return (outs[0], gets, lost) if reads is None else (outs[0], most[0])


@pytest.mark.parametrize("T,mfma,n_io,prefetch_n,shared", [
    (2, False, 0, 0, True), (64, True, 0, 0, True), (65, False, 2, 6, True), (130, True, 2, 6, False),
    (130, False, 0, 0, True)])
def test_one_pass_is_the_chunks(L, layer, monkeypatch, T, mfma, n_io, prefetch_n, shared):
    say("cached prompt", T, "mfma" if mfma else "octet", n_io, prefetch_n, shared)
    if mfma:
        monkeypatch.setenv("GLM53F_CACHE_MFMA", "1")
    sp, pool, W, B, sh = layer
    x = np.ascontiguousarray(S.x_host(sp, T, batch=4), np.float32)
    want, gets, _ = run(L, layer, x, sp.NE - 5, shared=shared)              # chunks: too few slots
    got, gets1, lost = run(L, layer, x, sp.NE + n_io + 64, n_io, prefetch_n, shared=shared)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert gets1 == gets and lost == 0
    sel = [0, T - 1]
    idx, _ = O.router(O.oracle(), x[sel], sp, W, B)
    mats = {int(e): pool[int(e) % NP] for e in np.unique(idx)}
    within(got[sel], O.moe(O.oracle(), x[sel], sp, W, B, mats, sh if shared else None)[0], f"T={T}")


def test_several_passes_are_the_chunks(L, layer):
    """More tokens than one planning pass takes: two passes, then one token that decodes."""
    say("cached prompt, several passes")
    sp = layer[0]
    x = np.ascontiguousarray(S.x_host(sp, 2048 + 129, batch=12), np.float32)
    want, gets, _ = run(L, layer, x, sp.NE - 5)
    got, gets1, lost = run(L, layer, x, sp.NE + 64)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert gets1 == gets and lost == 0


@pytest.mark.parametrize("mfma", [False, True])
def test_next_layer_prediction_in_a_pass(L, layer, monkeypatch, mfma):
    """Hints for the next layer from each chunk's own prediction, made inside the pass: the reads they start
    change nothing."""
    say("cached prompt, next layer predicted", "mfma" if mfma else "octet")
    if mfma:
        monkeypatch.setenv("GLM53F_CACHE_MFMA", "1")
    sp = layer[0]
    x = np.ascontiguousarray(S.x_host(sp, 130, batch=13), np.float32)
    want, gets, _ = run(L, layer, x, sp.NE - 5, n_io=2, prefetch_n=6, predict=True)
    got, gets1, lost = run(L, layer, x, 2 * sp.NE + 64, n_io=2, prefetch_n=6, predict=True)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert gets1 == gets and lost == 0


def test_failed_get_is_the_chunks_drop(L, layer):
    say("cached prompt with an expert that cannot be read")
    sp = layer[0]
    x = np.ascontiguousarray(S.x_host(sp, 130, batch=6), np.float32)
    want, _, lost = run(L, layer, x, sp.NE - 5, fails=(3, 17))
    got, _, lost1 = run(L, layer, x, sp.NE + 64, fails=(3, 17))
    assert lost1 == lost > 0
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_gets_wait_for_hinted_reads(L, layer):
    """A cold cache with hints: at most top-k reads of the call's own are under way at a time beside the
    prefetch's n_io, so that the hinted reads are not overtaken."""
    say("cached prompt, cold with hints")
    sp, pool = layer[:2]
    x = np.ascontiguousarray(S.x_host(sp, 64, batch=10), np.float32)
    want, _, _ = run(L, layer, x, sp.NE - 5)
    mem = []

    def pinned(a):                                   # copies from other memory are not asynchronous
        mem.append(L.g53h_host_alloc(a.nbytes))
        b = np.frombuffer((C.c_uint8 * a.nbytes).from_address(mem[-1]), a.dtype)
        b[:] = a
        return b
    try:
        pool = [[(pinned(w), pinned(s)) for w, s in mats] for mats in pool]
        got, most = run(L, (sp, pool) + layer[2:], x, sp.NE + 64, n_io=2, prefetch_n=6, reads=[])
    finally:
        for m in mem:
            L.g53h_host_free(m)
    assert 0 < most <= sp.K + 2
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_pass_needs_memory_only_for_what_is_not_held(L):
    """A call that cannot take the pass (too few slots) leaves no claim on memory: when HBM is full at the
    next call, which could take it, the chunks run; with room again the pass does. Same output each time."""
    say("cached prompt, HBM full")
    sp = S.spec(2, NE=24, K=16, seed=8)              # the largest workspace: 2000 tokens, top-16
    layer = sp, [S.expert_host(sp, p) for p in range(NP)], S.router_host(sp), S.bias_host(sp), S.expert_host(sp, "shared")
    x = np.ascontiguousarray(S.x_host(sp, 2000, batch=9), np.float32)
    one = glm53h.G53hExpert()
    g = glm53h.G53hMoeLayer(hidden=sp.E, inter=sp.I, n_experts=sp.NE, topk=sp.K, router_dt=1, block_c=128,
                            shared=C.addressof(one))
    growth = L.g53h_grouped_growth
    growth.argtypes, growth.restype = [C.POINTER(glm53h.G53hMoeLayer), C.c_int], C.c_size_t
    if growth(C.byref(g), x.shape[0]) == 0:
        pytest.skip("the library holds a larger workspace already")
    want, _, _ = run(L, layer, x, sp.NE - 5)
    was = L.g53h_set_mem_free(32 << 20)
    try:
        got, _, _ = run(L, layer, x, sp.NE + 64)
    finally:
        L.g53h_set_mem_free(was)
    assert growth(C.byref(g), x.shape[0]) > 0        # no pass of all tokens was made
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    got, _, _ = run(L, layer, x, sp.NE + 64)
    assert growth(C.byref(g), x.shape[0]) == 0
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def holds(layer, expert, at_hint=False):
    """A caller's own hold on an expert, as include/glm53f.h allows: taken before the calls, or by another
    user of the cache while a call runs (in its first hint)."""
    def hold(c):
        ref, taken = C.pointer(c.src), []

        def take(*_):
            if not taken:
                taken.append(c.src.get(ref, layer, expert, C.byref(glm53h.Glm53fExpertQ())))
        hint = glm53h.HINT_FN(take)
        if at_hint:
            c.src.hint = hint
        else:
            take()

        def release(_hint=hint):
            assert taken == [0]
            c.src.release(ref, layer, expert)
        return release
    return hold


@pytest.mark.parametrize("mfma", [False, True])
@pytest.mark.parametrize("where", ["other layer", "this layer", "during the call"])
def test_held_slots_leave_room(L, layer, monkeypatch, where, mfma):
    """As many slots as experts, one of them held by the caller: no expert is dropped and the output is that
    of the chunks."""
    say("cached prompt, a slot held", where, "mfma" if mfma else "octet")
    if mfma:
        monkeypatch.setenv("GLM53F_CACHE_MFMA", "1")
    sp = layer[0]
    x = np.ascontiguousarray(S.x_host(sp, 64, batch=7), np.float32)
    want, _, _ = run(L, layer, x, sp.NE - 5)
    hold = holds(0 if where == "this layer" else 1, 3, at_hint=where == "during the call")
    got, _, lost = run(L, layer, x, sp.NE, prefetch_n=6, hold=hold)
    assert lost == 0
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("T", [1, 3])
def test_int4_shared_expert_beside_mfma_slots(L, layer, monkeypatch, T):
    """A shared expert that cannot be kept tiled: the row kernels read the MFMA-tiled views as rows, and the
    output is that of row-major slots."""
    say("cached, int4 shared expert", T)
    sp, pool, W, B, sh = layer
    keep = [dev_quant(w, s, r, c, 128, 128) + (r, c) for (w, s), (r, c) in
            zip(sh, [(sp.I, sp.E), (sp.I, sp.E), (sp.E, sp.I)])]
    layer = sp, pool, W, B, [imat(*k) for k in keep]
    x = np.ascontiguousarray(S.x_host(sp, T, batch=11), np.float32)
    monkeypatch.setenv("GLM53F_CACHE_ROWMAJOR", "1")
    want, _, _ = run(L, layer, x, sp.NE)
    monkeypatch.delenv("GLM53F_CACHE_ROWMAJOR")
    monkeypatch.setenv("GLM53F_CACHE_MFMA", "1")
    got, _, _ = run(L, layer, x, sp.NE)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
