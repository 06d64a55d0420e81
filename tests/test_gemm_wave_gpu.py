"""The tolerance GEMM whose weights travel wave by wave (krasis_amd/csrc/kr_prefill_w.hip, tiles of 96 rows) against the register-staged kernels (kr_prefill_h.hip): the same
fragments in the same order per sum, so the outputs are compared bit for bit.  kr_moe_set_gemm_mode: 1 = the default dispatch, 3 = register-staged kernels only; a store's option gemm_ring: 1, 0."""
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


@pytest.mark.parametrize("kinds,kw,n_tok", [
    (["la", "gqa"], dict(la_heads=(14, 28), la_dkdv=(128, 128), nh=8), 500),      # 10752 + 56 columns: six panels of eight column blocks, the sixth over the border; a second matrix that is no whole wave; 258 tiles, 6 row tiles of which the last has 20 rows
    (["la", "gqa"], dict(la_heads=(16, 32), la_dkdv=(128, 128), nh=8), 450),      # 12288 + 64
    (["la", "gqa"], dict(la_heads=(9, 27), la_dkdv=(128, 128), nh=8), 600),        # 9216 + 54: rows of the second result that are no whole 16-byte pieces; 259 tiles, a last row tile of 24 rows
    (["gqa", "la"], dict(nh=32), 700),                                             # q with its gate, k and v: 8192 + 256 + 256 columns, two borders inside the fifth panel; 272 tiles, a last row tile of 28 rows
])
def test_several_matrices_of_a_launch(kinds, kw, n_tok):
    """the projections of one input are one launch of up to three matrices: the last position's logits, and every layer's caches and states, after prompts whose launches have 220 tiles and more"""
    from tests.test_decode_gpu import build
    rng = np.random.default_rng(n_tok)
    res = []
    for form in (0, 1):
        st, eng, orc, keep, d = build(seed=41, kv_max=n_tok + 8, kinds=kinds, hd=128, **kw)
        st.set_attention_mode(True, gemm_fast=True)
        st.set_option("gemm_ring", form)
        if not res:
            toks = [int(t) for t in rng.integers(0, d["V"], n_tok)]
        lg = np.empty(d["V"], np.float32)
        st.prefill(toks, 0, lg.ctypes.data)
        out = [lg.view(np.uint32)]
        for li, kind in enumerate(d["kinds"]):
            if kind == "gqa":
                k = np.empty((d["kv_max"], d["nkv"] * d["hd"]), np.uint16); v = np.empty_like(k)
                st.get_decode_state(li, k, v, None, None)
                out += [k[:n_tok], v[:n_tok]]
            else:
                cs = np.empty(d["conv_dim"] * 4, np.float32); rs = np.empty(d["nv"] * d["dk"] * d["dv"], np.float32)
                st.get_decode_state(li, None, None, cs, rs)
                out += [cs.view(np.uint32), rs.view(np.uint32)]
        assert np.isfinite(lg).all()
        res.append(out)
    for a, b in zip(*res):
        assert np.array_equal(a, b)
