"""Steps of one token per request through the recurrent mixers, scan and output in one launch (sv_lin_step_kernel in csrc/kr_serve_ops.hip), against the float64 restatements.

Sizes: the three key widths that launch takes and two beside them, value widths of one wave and of eight, whole and ragged; a request's first token, and requests that end and begin
on the way.  Tolerance: that of the f32 store's other tests (2e-4 of the stream's scale)."""
import numpy as np
import pytest

from tests import oracle_gasavik as G
from tests import oracle_lufozen as L
from tests import oracle_midisun as M
from tests import test_gasavik_gpu, test_lufozen_gpu, test_midisun_gpu
from tests.test_midisun_gpu import rel

pytestmark = pytest.mark.gpu

MIXERS = [(M, M.retention(2, 128, 128, [0.9, 0.999], rot_dims=64)), (M, M.retention(3, 32, 7, [0.5, 0.9, 1.0])), (M, M.retention(1, 64, 72, [0.97], rot_dims=6)),
          (M, M.retention(1, 64, 129, [0.97])), (M, M.retention(2, 36, 16, [0.9, 0.8])),
          (M, M.mlstm(2, 128, 128)), (M, M.mlstm(3, 32, 17, gate_cap=0.7)), (M, M.mlstm(1, 64, 100)),
          (L, L.gla(2, 128, 128)), (L, L.gla(1, 32, 9)), (L, L.gla(2, 64, 40)),
          (G, G.wkv(2, 32)), (G, G.wkv(1, 128)), (G, G.wkv(2, 64)),
          (G, G.delta(4, 2, 128, 128, 4)), (G, G.delta(2, 1, 32, 20, 2)), (G, G.delta(2, 2, 64, 64, 3))]


@pytest.mark.parametrize("O,mixer", MIXERS)
def test_token_by_token(O, mixer):
    cfg = O.make_config(width=64, vocab=50, layers=[O.layer(mixer, O.dense(24))] * 2)
    W = O.random_weights(cfg, 5)
    eng = {M: test_midisun_gpu, L: test_lufozen_gpu, G: test_gasavik_gpu}[O].engine(cfg, W)
    rng = np.random.default_rng(6)
    seqs = [[int(t) for t in rng.integers(0, 50, 36)] for _ in range(3)]
    ref = [O.forward(cfg, W, s)[0] for s in seqs]
    rows = [[], [], []]
    for i in range(36):                                       # the last request begins at token 0 when the others are at 9, and a slot is given back and taken again
        live = [(r, seqs[r][j]) for r, j in ((0, i), (1, i), (2, i - 9)) if j >= 0]
        if i == 20:
            eng.finish(1); rows[1] = []
        if i >= 20:
            live[1] = (1, seqs[1][i - 20])
        for (r, _), l in zip(live, eng.step([(r, [t], [0]) for r, t in live])[0]):
            rows[r].append(l)
    for r in range(3):
        assert rel(np.stack(rows[r]), ref[r][:len(rows[r])]) < 2e-4, r
