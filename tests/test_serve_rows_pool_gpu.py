"""Logits that a step stores in the caller's own memory (kr_serve_rows_alloc): arrays stay what they were while others are made, blocks come round again, and what has no block -- more
than the pool holds, rows past its largest block, memory of the caller's -- takes the copy."""
import ctypes as C
import gc
import os
import threading

import numpy as np
import pytest

from krasis_amd import serve_store as S
from krasis_amd._lib import check_serve
from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


def model(vocab=4099):
    return O.make_config(width=64, vocab=vocab, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 1, 0, scale=0.3), "mlp": O.moe(4, 2, 1, 1, 32, 2.0, 32, 2.0)}])


def run(eng, rid, toks):
    """the prompt and single tokens, which replay a captured step from the third on"""
    out = [eng.step([(rid, toks[:20], [3, 19])])[0]]
    out += [eng.step([(rid, [t], [0])])[0] for t in toks[20:]]
    eng.finish(rid)
    return out


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_arrays_keep_their_values_and_blocks_return(dtype, monkeypatch):
    cfg = model(); W = O.random_weights(cfg, 3); toks = tokens(cfg, 32, 4)
    eng = engine(cfg, W, dtype, max_tokens=512)
    monkeypatch.setattr(eng.store._rows, "take", lambda *a: None)
    ref = run(eng, "copied", toks)
    monkeypatch.undo()
    kept = [run(eng, i, toks) for i in range(3)]
    assert eng.store.graph_replays() > 0
    for got in kept:
        for a, b in zip(got, ref):
            assert a.dtype == np.float32 and a.shape == b.shape and a.flags.writeable and a.flags.c_contiguous
            assert np.array_equal(a, b)
    views = [g[1][:, 5:9] for g in kept]                 # a view holds its block
    before = [v.copy() for v in views]
    kept = None; gc.collect()
    used = eng.store._rows._bytes
    for _ in range(40):
        run(eng, "again", toks)
    assert eng.store._rows._bytes == used                # blocks came round
    assert all(np.array_equal(v, b) for v, b in zip(views, before))
    last = eng.step([("z", toks[:5], [4])])[0]
    want = last.copy()
    eng.store.close()
    assert np.array_equal(last, want) and all(np.array_equal(v, b) for v, b in zip(views, before))
    last[:] = 0


def test_past_the_pool_and_past_its_blocks(monkeypatch):
    monkeypatch.setattr(S._RowPool, "MOST", 1 << 20)
    monkeypatch.setattr(S._RowPool, "LARGEST", 256 << 10)
    cfg = model(); W = O.random_weights(cfg, 5); toks = tokens(cfg, 40, 6)
    eng = engine(cfg, W, "bfloat16", max_tokens=512)
    ref = eng.step([("a", toks, [39])])[0].copy()
    held = []
    for i in range(70):                                  # 64 KB each: the pool is full after sixteen
        eng.finish("a"); held.append(eng.step([("a", toks, [39])])[0])
    assert eng.store._rows._bytes <= 1 << 20
    assert all(np.array_equal(h, ref) for h in held)
    eng.finish("a")
    rows = eng.step([("a", toks, list(range(40)))])[0]   # 656 KB: no block
    assert rows.base is None
    eng.finish("a")
    monkeypatch.setattr(S._RowPool, "LARGEST", 1 << 20); monkeypatch.setattr(S._RowPool, "MOST", 4 << 20)
    assert np.array_equal(eng.step([("a", toks, list(range(40)))])[0], rows)      # the same launches into a block


def test_rows_of_the_c_interface():
    cfg = model(); W = O.random_weights(cfg, 7); toks = np.asarray(tokens(cfg, 9, 8), np.int32)
    eng = engine(cfg, W, "bfloat16", max_tokens=512)
    st, lib = eng.store, eng.store._lib
    rows, V = 3, cfg["vocab"]
    p = C.c_void_p()
    check_serve(lib.kr_serve_rows_alloc(st._h, 1 << 20, C.byref(p)))
    whole = np.frombuffer((C.c_float * (1 << 18)).from_address(p.value), np.float32)
    want = np.asarray([0, 4, 8], np.int32); amax = np.empty(rows, np.int32)
    ref = None
    for at in (0, 4, 1, (1 << 18) - rows * V + 1):       # aligned; aligned; not to 16 bytes: copied; past the end: an ordinary destination has to hold it
        slot = st.admit()
        dst = whole[at:at + rows * V] if at + rows * V <= whole.size else np.empty(rows * V, np.float32)
        whole[:] = -1.0
        slots, counts = np.asarray([slot], np.int32), np.asarray([9], np.int32)
        check_serve(lib.kr_serve_step(st._h, 1, slots.ctypes.data, counts.ctypes.data, toks.ctypes.data, rows, want.ctypes.data, dst.ctypes.data, amax.ctypes.data))
        ref = dst.copy() if ref is None else ref
        assert np.array_equal(dst, ref) and np.array_equal(amax, ref.reshape(rows, V).argmax(1))
        if at < 1 << 17:
            assert np.all(whole[:at] == -1.0) and np.all(whole[at + rows * V:] == -1.0)
        st.release(slot)
    with pytest.raises(ValueError):
        check_serve(lib.kr_serve_rows_free(C.c_void_p(p.value + 64)))
    check_serve(lib.kr_serve_rows_free(p))
    with pytest.raises(ValueError):
        check_serve(lib.kr_serve_rows_free(p))
    with pytest.raises(ValueError):
        check_serve(lib.kr_serve_rows_alloc(st._h, 0, C.byref(p)))


def test_a_forked_child_reads_the_arrays():
    cfg = model(); W = O.random_weights(cfg, 11); toks = tokens(cfg, 28, 12)
    eng = engine(cfg, W, "bfloat16", max_tokens=512)
    held = run(eng, "a", toks)
    want = [h.copy() for h in held]
    pid = os.fork()
    if pid == 0:                                         # nothing of the device in here
        os._exit(0 if all(np.array_equal(h, w) for h, w in zip(held, want)) else 1)
    assert os.waitpid(pid, 0)[1] == 0
    assert all(np.array_equal(h, w) for h, w in zip(run(eng, "b", toks), want)) and all(np.array_equal(h, w) for h, w in zip(held, want))


def test_two_stores_on_two_threads():
    cfg = model(); W = O.random_weights(cfg, 9); toks = tokens(cfg, 28, 10)
    engs = [engine(cfg, W, "bfloat16", max_tokens=512) for _ in range(2)]
    ref = [a.copy() for a in run(engs[0], "r", toks)]
    bad, done = [], []

    def work(e):
        try:
            for i in range(30):
                if not all(np.array_equal(a, b) for a, b in zip(run(e, i, toks), ref)):
                    bad.append(i)
                done.append(e)
        except BaseException as err:                     # an exception would end its thread alone
            bad.append(err)
    ts = [threading.Thread(target=work, args=(e,)) for e in engs]
    for t in ts: t.start()
    for t in ts: t.join()
    assert not bad and [sum(d is e for d in done) for e in engs] == [30, 30], bad
