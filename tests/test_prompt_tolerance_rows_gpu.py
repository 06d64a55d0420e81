"""Launches of the tolerance prompt pass that do the work of two (krasis_amd/csrc/kr_prefill_ops.hip), and the pair sort of long chunks (kr_prefill.hip), against the launches that they
stand for: bit for bit, since the order of every sum is the same.  And the strips of the tolerance GEMM (kr_prefill_h.hip) against the exact form."""
import numpy as np
import pytest

from tests.test_gemm_fast_gpu import _setup
from tests.test_gemm_ring_gpu import _prefill_mode
from tests.util import rand_bf16

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.mark.parametrize("la_heads,ntok", [((1, 2), 65), ((2, 4), 300), ((4, 32), 130), ((8, 40), 70)])      # rows of 256, 512, 4096 (two pieces a thread, all of them) and 5120 values
def test_gated_norm_leaves_the_row_image(la_heads, ntok):
    from tests.test_attn_fast_gpu import build
    toks, res = None, []
    for fused in (0, 1):
        st, eng, orc, keep, d = build(seed=37, kv_max=400, kinds=["la", "la"], la_heads=la_heads)
        st.set_attention_mode(True, gemm_fast=True)
        st.set_option("norm_rows", fused)
        if toks is None:
            toks = [int(t) for t in np.random.default_rng(9).integers(0, d["V"], ntok)]
        lg = np.empty(d["V"], F)
        st.prefill(toks, 0, lg.ctypes.data)
        res.append(lg)
    assert np.isfinite(res[1]).all()
    assert np.array_equal(res[0].view(np.uint32), res[1].view(np.uint32)), float(np.abs(res[0] - res[1]).max())


@pytest.mark.parametrize("E,k,M", [(8, 8, 4200), (65, 10, 3300), (512, 10, 3400)])      # more than 32768 pairs: rows and tiles by wave scans; one wave, one expert in the second, eight waves
def test_pair_sort_of_long_chunks(E, k, M):
    eng, experts, shared, rng, torch = _setup(256, 128, E, k, 0, 1.0)
    x = rand_bf16(rng, (M, 256))
    ids = np.argsort(rng.random((M, E)), axis=1)[:, :k].astype(np.int32)
    ids[5, 1] = -1; ids[9, :] = -1
    if E > 64:
        ids[ids == 3] = 64 if E == 65 else 63                     # an expert without rows, another with twice its share
    w = rng.random((M, k)).astype(F)
    whole = _prefill_mode(eng, torch, x, ids, w, 0)
    h = M // 2
    parts = np.concatenate([_prefill_mode(eng, torch, x[:h], ids[:h], w[:h], 0), _prefill_mode(eng, torch, x[h:], ids[h:], w[h:], 0)])
    assert np.array_equal(whole.view(np.uint32), parts.view(np.uint32)), float(np.abs(whole - parts).max())


@pytest.mark.parametrize("H,I,E,k,M", [
    (2048, 512, 64, 10, 64),       # ten rows an expert: tiles of up to 16 and second ones
    (256, 128, 8, 2, 1),           # one row; one step a strip
    (384, 128, 8, 2, 17),          # an odd group count: the last step of a strip holds one group
    (512, 384, 300, 4, 1050),      # hundreds of experts: fourteen rows each; an odd group count in the down projection, strips that do not fill a workgroup
])
def test_strips_of_few_rows_per_expert(H, I, E, k, M):
    """Rows and hidden values are rounded to f16 once each, relative error at most 2^-11 a value, in both products of an expert: the norm of the difference to the exact form (sixteen
    times finer digits) stays under 2 * 2^-11."""
    eng, experts, shared, rng, torch = _setup(H, I, E, k, 0, 1.0)
    x = rand_bf16(rng, (M, H))
    ids = np.argsort(rng.random((M, E)), axis=1)[:, :k].astype(np.int32)
    if M > 16:
        ids[:16, 0] = 0; ids[3, 1] = -1; ids[7, :] = -1                # an expert that fills its tile, rows left out
        ids[:16, 1:][ids[:16, 1:] == 0] = -1
    w = rng.random((M, k)).astype(F)
    exact, fast = (_prefill_mode(eng, torch, x, ids, w, mode) for mode in (0, 1))
    rel = float(np.linalg.norm((fast - exact).astype(np.float64)) / np.linalg.norm(exact.astype(np.float64)))
    assert np.isfinite(fast).all() and 0 < rel <= 2.0 ** -10, rel
    if M > 16:
        assert not fast[7].any()
