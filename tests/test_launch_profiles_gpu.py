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
