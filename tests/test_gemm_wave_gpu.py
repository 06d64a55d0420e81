"""The tolerance GEMM whose weights travel wave by wave (krasis_amd/csrc/kr_prefill_w.hip, tiles of 96 rows) against the register-staged kernels (kr_prefill_h.hip): the same
fragments in the same order per sum, so the outputs are compared bit for bit.  kr_moe_set_gemm_mode: 1 = the default dispatch, 3 = register-staged kernels only."""
import numpy as np
import pytest

from tests.test_gemm_fast_gpu import _setup
from tests.test_gemm_ring_gpu import _prefill_mode
from tests.util import rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,E,k,M,n_shared", [
    (128, 128, 32, 2, 330, 0),         # one group of 128: two lines of k; tiles of one row block
    (256, 384, 8, 2, 256, 0),          # one stage; an odd number of groups behind a whole stage in the second product; tiles of two row blocks
    (384, 256, 6, 6, 97, 0),           # every expert one row past a tile; 384 columns: waves without columns beside waves with whole ones
    (640, 128, 6, 6, 96, 0),           # whole tiles
    (512, 640, 2, 2, 289, 0),          # several tiles an expert, a last one of one row
    (2048, 512, 32, 10, 300, 0),       # eight stages
    (256, 1408, 4, 2, 3100, 1),        # dense: gate and up of the shared expert, 33 row tiles of which the last has 28 rows
])
def test_wave_gemm_bit_identical_to_register_staged(H, I, E, k, M, n_shared):
    eng, experts, shared, rng, torch = _setup(H, I, E, k, n_shared, 2.0 if n_shared else 1.0)
    x = rand_bf16(rng, (M, H)); ids = np.stack([rng.choice(E, k, replace=False) for _ in range(M)]).astype(np.int32)
    if E not in (2, 6):
        ids[3, 1] = -1; ids[7, :] = -1
    w = rng.random((M, k)).astype(np.float32)
    staged = _prefill_mode(eng, torch, x, ids, w, 3)
    for _ in range(3):
        got = _prefill_mode(eng, torch, x, ids, w, 1)
        assert np.isfinite(got).all()
        assert np.array_equal(staged.view(np.uint32), got.view(np.uint32)), float(np.abs(staged - got).max())
