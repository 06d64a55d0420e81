"""The measurement hooks time the launches that a call without them makes."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gemm_fast_gpu import _setup
from tests.test_prefill_strips_gpu import _forward
from tests.util import rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,sums", [(1, 0), (2, 3)])
def test_expert_operator(M, sums):
    """one row: its sum leaves the down projection, so there is no launch of the third kind"""
    from krasis_amd._lib import check
    eng, experts, shared, rng, torch = _setup(256, 128, 8, 3)
    x = rand_bf16(rng, (M, 256)); ids = np.stack([rng.choice(8, 3, replace=False) for _ in range(M)]).astype(np.int32); w = rng.random((M, 3)).astype(np.float32)
    plain = _forward(eng, torch, x, ids, w)
    check(eng._lib.kr_set_profiling(eng._h, 1))
    timed = [_forward(eng, torch, x, ids, w) for _ in range(3)]
    ms, n = C.c_double(), C.c_long()
    seen = []
    for kind in range(3):
        check(eng._lib.kr_get_profile(eng._h, kind, C.byref(ms), C.byref(n)))
        seen.append(n.value)
        assert (ms.value > 0) == (n.value > 0)
    check(eng._lib.kr_set_profiling(eng._h, 0))
    assert seen == [3, 3, sums]
    assert all(np.array_equal(t, plain) for t in timed)


def test_joined_decode_step():
    """attention beside the experts' gate and up product counts as the product; the merge of its shares, once there are several, as attention"""
    from tests import oracle_serve as O
    from tests.test_serve_gpu import engine, tokens
    cfg = O.make_config(width=128, vocab=70, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(8, 2, 64, 64, 0, 64, scale=0.1), "mlp": O.moe(8, 3, 1, 1, 96, 1.5, 64, 2.0)}])
    W = O.random_weights(cfg, 31)
    eng = engine(cfg, W, "bfloat16")
    a = tokens(cfg, 620, 32)
    eng.step([("a", a[:100], [])])
    seen = []
    for i, n in ((100, 101), (101, 600), (600, 601)):
        eng.store.set_profiling(n - i == 1)
        eng.step([("a", a[i:n], [0])])
        seen.append(eng.store.profile())
    eng.store.set_profiling(False)
    assert seen[0][1] > 0 and seen[0][3] == 0 and seen[0][4] > 0
    assert seen[2][1] > 0 and seen[2][3] > 0 and seen[2][4] > 0
