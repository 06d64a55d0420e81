"""How a prompt is cut into chunks by default (csrc/kr_decode_prefill.cpp: prompt_chunk): as few of at most 4096 tokens as hold it where attention runs in the tolerance form, but at
least two from 1025 tokens on where a layer is MLA or holds native GGUF experts, and three from 4609 to 7680 where one is MLA; about 1024 tokens each in the exact form."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def store(kind):
    if kind == "mla":
        from tests.test_mla_gpu import build
        return build(kv_max=1200)
    from tests.test_decode_gpu import build
    return build(kv_max=1200, gguf=kind == "gguf")


@pytest.mark.parametrize("kind,two", [("plain", False), ("gguf", True), ("mla", True)])
def test_tokens_per_chunk(kind, two):
    st, eng, orc, keep, d = store(kind)
    got = ctypes.c_int(0)

    def chunk(n):
        assert st._lib.kr_decode_prefill_chunk(st._h, n, ctypes.byref(got)) == 0
        return got.value

    exact = [(1, 1), (777, 777), (1025, 513), (3072, 1024), (8192, 1366)]
    for n, want in exact:
        assert chunk(n) == want, n
    for fast in (False, True):
        st.set_attention_mode(True, gemm_fast=fast)
        for n, want in [(1, 1), (1024, 1024), (1025, 576 if two else 1025), (2048, 1024 if two else 2048), (4096, 2048 if two else 4096), (4097, 2112), (4608, 2304), (4609, 1600 if kind == "mla" else 2368), (7680, 2560 if kind == "mla" else 3840), (7681, 3904), (8192, 4096), (8193, 2752)]:
            assert chunk(n) == want, (n, fast)
    st.set_prefill_chunk(64)
    assert chunk(1) == 1 and chunk(2048) == 64
    st.set_attention_mode(False)
    assert chunk(2048) == 64
    for n in (0, -1):
        assert st._lib.kr_decode_prefill_chunk(st._h, n, ctypes.byref(got)) != 0


def test_the_default_cut_is_the_one_stated():
    """1100 tokens of an MLA store: the bits of the same prompt with 576 tokens per chunk asked for"""
    st, eng, orc, keep, d = store("mla")
    toks = [int(t) for t in np.random.default_rng(3).integers(0, d["V"], 1100)]
    st.set_attention_mode(True, gemm_fast=True)
    out = []
    for chunk in (0, 576):
        st.set_prefill_chunk(chunk)
        out.append(np.empty(d["V"], F))
        st.prefill(toks, 0, out[-1].ctypes.data)
    assert np.isfinite(out[0]).all() and np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
