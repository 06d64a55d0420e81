"""The serving store's row kernels (embedding with the first norm, residual sum with the next norm, logits' norm) where their forms meet: widths that are no multiples of four or pass
16384 take the scalar kernels, others a row in registers by 256, 512 or 1024 threads; up to 64 rows are spread wider.  And the greedy token at vocabularies of both forms."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, rel, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [4, 66, 1024, 1028, 2048, 2052, 4096, 4100, 16384, 16388])
@pytest.mark.parametrize("n", [1, 64, 65])
def test_rows_of_a_layer(width, n):
    mixer = O.attn(1, 1, 8, 8, 0, 4, scale=0.3)
    cfg = O.make_config(width=width, vocab=41, eps=1e-5, layers=[{"type": "attention", "mixer": mixer, "mlp": O.dense(8)}, {"type": "attention", "mixer": mixer, "mlp": O.moe(3, 2, 1, 1, 8, 1.5, 8, 1.0)}])
    W = O.random_weights(cfg, 41, router_gain=40.0); toks = tokens(cfg, n, 42)
    logits, ref = O.forward(cfg, W, toks)
    eng = engine(cfg, W)
    eng.store.set_capture(True)
    got, _ = eng.step([("a", toks, [n - 1])])
    cap = eng.store.read_capture(n)
    # one f32 rounding per operand over sums of `width` terms: 6e-8 sqrt(16384) = 8e-6 relative to the row, with room for the layer's few such sums
    assert rel(cap[0], ref[0]) < 1e-4 and rel(cap[1], ref[1]) < 1e-4
    assert rel(got, logits[n - 1:]) < 2e-4


@pytest.mark.parametrize("vocab", [3, 4, 4095, 4096, 4100, 12300])
def test_greedy_token(vocab):
    cfg = O.make_config(width=32, vocab=vocab, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(1, 1, 8, 8, 0, 4, scale=0.3), "mlp": O.dense(8)}])
    W = O.random_weights(cfg, 43); toks = tokens(cfg, 5, 44)
    best = int(np.argmax(O.forward(cfg, W, toks)[0][4]))
    for twin in (best - 1, best + 1):                                     # a tie: the lowest index wins
        if 0 <= twin < vocab:
            W["head"][twin] = W["head"][best]
    logits, amax = engine(cfg, W).step([("a", toks, [4])])
    assert int(amax[0]) == int(logits.argmax(-1)[0]) == max(best - 1, 0)
