"""Where a step wants every row in its place, the sum that ends the last layer hands on the final norm's rows (csrc/kr_serve.cpp): the same bits as the norm's own launch, which takes the rows
in any other order; rows of one and several chunks a thread, widths of neither kernel's; and the two kinds of steps in turn, until both are replayed from graphs."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


def config(width, mlp):
    return O.make_config(width=width, vocab=300, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 32, 32, 0, 16, scale=0.3), "mlp": m} for m in (None, mlp)])


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("width,mlp", [(64, O.dense(64)), (2080, None), (4128, O.dense(32)), (36, O.dense(36)), (128, O.moe(4, 2, 1, 1, 32, 2.0, 32, 2.0))])
def test_rows_in_place_equal_rows_in_any_order(width, mlp, dtype):
    cfg = config(width, mlp); W = O.random_weights(cfg, 71)
    eng = engine(cfg, W, dtype)
    for n in (1, 2, 64, 65, 200):
        toks = tokens(cfg, n, 72)
        a, am = eng.step([("a", toks, list(range(n)))])
        b, bm = eng.step([("b", toks, list(range(n))[::-1] if n > 1 else [0, 0])])
        eng.finish("a"); eng.finish("b")
        assert np.array_equal(a, b[::-1][:n]) and np.array_equal(am, bm[::-1][:n]), n


def test_both_kinds_of_steps_in_turn():
    cfg = config(64, O.dense(64)); W = O.random_weights(cfg, 73)
    toks = tokens(cfg, 64, 74)
    eng, ref = engine(cfg, W), engine(cfg, W)
    ref.store.set_capture(True)                                          # eager
    for i in range(24):
        places = ([0], [0]) if i % 3 else ([0, 0], [])                   # as many wanted rows either way
        got, want = (e.step([("a", [toks[i]], places[0]), ("b", [toks[63 - i]], places[1])]) for e in (eng, ref))
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), i
    assert eng.store.graph_replays() > 8
