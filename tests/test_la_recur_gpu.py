"""The exact delta rule at the edges of its blocks: blocks of sixteen tokens, sixteen columns per workgroup, eight lanes per column.  Bit for bit against the token-by-token decode and the
oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_decode_gpu import build
from tests.test_prefill_model_gpu import _snapshot
from tests.test_standalone_ops_gpu import ptr, store

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("n_tok", [2, 15, 16, 17, 31, 32, 33, 50])
def test_blocks_of_tokens(n_tok):
    st, eng, orc, keep, d = build(kv_max=64)
    toks = [int(x) for x in np.random.default_rng(n_tok).integers(0, d["V"], n_tok)]
    want, got = np.empty(d["V"], F), np.empty(d["V"], F)
    for i, t in enumerate(toks):
        st.decode_step(t, i, want.ctypes.data)
    state = _snapshot(st, d)
    d["reset"]()
    st.prefill(toks, 0, got.ctypes.data)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    for a, b in zip(_snapshot(st, d), state):
        assert all(x.tobytes() == y.tobytes() for x, y in zip(a, b))


@pytest.mark.parametrize("nv,dk,dv", [(1, 64, 64), (3, 64, 72), (2, 64, 248), (1, 64, 256), (1, 128, 128), (3, 128, 136), (2, 128, 256)])
def test_columns(nv, dk, dv):
    rng = np.random.default_rng(nv + dv)
    q, k = (rng.standard_normal(nv * dk).astype(F) for _ in range(2))
    v = rng.standard_normal(nv * dv).astype(F); g = -rng.random(nv).astype(F); beta = rng.random(nv).astype(F)
    state = (rng.standard_normal(nv * dk * dv) * 0.1).astype(F); out = np.empty(nv * dv, F)
    dev = state.copy()
    store().linear_attention_recurrent(ptr(dev), ptr(q), ptr(k), ptr(v), ptr(g), ptr(beta), ptr(out), nv, dk, dv)
    ref, after = O.la_recurrent(state, q, k, v, g, beta, nv, dk, dv)
    assert np.asarray(out, F).tobytes() == np.asarray(ref, F).tobytes() and dev.tobytes() == np.asarray(after, F).tobytes()
