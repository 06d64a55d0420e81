"""The serving store's expert choice where its forms meet: one wave's registers hold up to 64 and 128 experts, more go through LDS; up to 16 tokens are sorted in the same launch, up to
1024 pairs in one workgroup, more in blocks of 2048.  f32 store, so that the oracle's choices are the store's."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, rel, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,top,groups,keep", [(2, 1, 1, 1), (63, 5, 1, 1), (64, 6, 4, 2), (65, 64, 1, 1), (126, 3, 63, 2), (128, 8, 64, 63), (129, 7, 3, 2), (200, 2, 1, 1)])
@pytest.mark.parametrize("n", [1, 16, 17])
def test_choice_and_rows(experts, top, groups, keep, n):
    cfg = O.make_config(width=32, vocab=40, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 0, 4, scale=0.3), "mlp": O.moe(experts, top, groups, keep, 8, 1.5)}])
    W = O.random_weights(cfg, 31)
    W["l0.mlp.router"][1::2] = W["l0.mlp.router"][:experts // 2 * 2:2]      # neighbours score alike: the lower index has to win
    toks = tokens(cfg, n, 32)
    ref = O.forward(cfg, W, toks)[1][0]
    eng = engine(cfg, W)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    assert rel(eng.store.read_capture(n)[0], ref) < 2e-4


@pytest.mark.parametrize("n,top", [(256, 4), (257, 4), (1025, 2), (700, 9)])
def test_rows_of_prompts(n, top):
    # 1024 pairs and one token more; several blocks of pairs, the last one ragged
    cfg = O.make_config(width=32, vocab=40, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 3, 4, scale=0.3), "mlp": O.moe(37, top, 1, 1, 8, 1.5, 8, 1.0)}])
    W = O.random_weights(cfg, 33); toks = tokens(cfg, n, 34)
    ref = O.forward(cfg, W, toks)[1][0]
    eng = engine(cfg, W, max_tokens=2048)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    assert rel(eng.store.read_capture(n)[0], ref) < 2e-4


@pytest.mark.parametrize("experts,groups,keep,top", [(12, 4, 3, 5), (96, 4, 3, 26), (132, 4, 3, 35)])
@pytest.mark.parametrize("n", [3, 40])
def test_groups_whose_score_is_minus_infinity(experts, groups, keep, top, n):
    # a correction of minus infinity takes experts out.  The sum of a group's two largest choice scores is minus infinity when one expert is left in it: such a group still
    # fills a free place among the kept ones (lowest index first), and its expert can be chosen
    from tests import oracle_midisun as M
    from tests.test_midisun_gpu import engine as midisun_engine
    cfg = M.make_config(64, 40, [M.layer(M.retention(2, 8, 8, (0.9, 0.95)), M.moe(experts, top, 16, groups, keep))], groups=1, taps=1)
    W = M.random_weights(cfg, 35)
    per = experts // groups
    for g in range(1, groups):
        W["l0.mlp.correction"][g * per:(g + 1) * per] = -np.inf
        W["l0.mlp.correction"][g * per + g % per] = 0.1 * g
    toks = tokens(cfg, n, 36)
    ref = M.forward(cfg, W, toks)[1][0]
    eng = midisun_engine(cfg, W)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    assert rel(eng.store.read_capture(n)[0], ref) < 2e-4
