"""The last tile of a product takes only the row blocks it has (csrc/kr_serve_tile.hip): every number of them in the 256-row tile of a bf16 store and the 128-row tiles of both
types, one row to either side of each border, against float64.  Bounds: test_serve_gemm_gpu.py (bf16 rounding of the rows, f32 sums)."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gemm_gpu import stream_model
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,full,vocab,rests", [("bfloat16", 2048, 7168, (1, 64, 65, 128, 129, 192, 193)), ("bfloat16", 384, 4224, (1, 64, 65)), ("float32", 1024, 4100, (1, 64, 65))])
def test_rows_of_the_last_tile(dtype, full, vocab, rests):
    cfg = stream_model(64, vocab); W = O.random_weights(cfg, 31)
    head = W["head"].astype(np.float64)
    toks = tokens(cfg, full + max(rests), 32)
    eng = engine(cfg, W, dtype, max_tokens=4096)
    eng.store.set_capture(True)
    for rest in rests:
        n = full + rest
        logits, amax = eng.step([("a", toks[:n], list(range(n)))])
        x = eng.store.read_capture(n)[-1].astype(np.float64)
        eng.finish("a")
        h = O.layer_norm(x, W["final.norm"].astype(np.float64), W["final.norm.b"].astype(np.float64), 1e-5)
        spread = np.sqrt(((np.abs(h) * (2.0 ** -9 if dtype == "bfloat16" else 0.0)) ** 2) @ (head.T ** 2))
        assert np.all(np.abs(logits - h @ head.T) <= 6.0 * spread + 1e-5 * np.abs(h) @ np.abs(head.T)), rest
        assert np.array_equal(amax, logits.argmax(-1))
