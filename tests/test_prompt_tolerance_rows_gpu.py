"""Launches of the tolerance prompt pass that do the work of two (krasis_amd/csrc/kr_prefill_ops.hip), and the pair sort of long chunks (kr_prefill.hip), against the launches that they
stand for: bit for bit, since the order of every sum is the same."""
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
