"""Decode steps whose dense feed-forward, and whose mixer projections with the residual gate's, are strips of one launch (csrc/kr_serve_skinny.hip): a bf16 store against the f32
store of the same weights, which other tests hold to the float64 restatement.

The sizes are the edges of that launch: one row to sixteen and the next one, one and several strips of pairs, a feed-forward width that the strips do not take, columns behind the
pairs or none, biases, the other activation.  Tolerance: that of the store's other bf16 tests (rows rounded to eight bits before every product; test_midisun_gpu.py)."""
import numpy as np
import pytest

from tests import oracle_midisun as O
from tests.test_midisun_gpu import tokens

pytestmark = pytest.mark.gpu


def stores(cfg, W, change):
    from krasis_amd import model_registry as R
    from krasis_amd.scheduler import BatchEngine
    for dtype in ("float32", "bfloat16"):
        spec = R.midisun_spec(cfg)
        change(spec)
        eng = BatchEngine(spec, dtype=dtype, max_tokens=2048, max_slots=17)
        eng.load_arrays(W)
        yield eng


@pytest.mark.parametrize("requests,width,ff,bias,gate,act", [
    (1, 64, 32, False, True, None), (2, 128, 96, True, True, None), (15, 64, 224, False, False, None), (16, 96, 160, True, False, "ACT_GELU_TANH"), (16, 64, 32, True, True, None),
    (17, 64, 96, True, True, None), (3, 64, 48, True, True, None), (4, 2048, 4128, True, True, "ACT_GELU_TANH"),
])
def test_steps_close_to_the_f32_store(requests, width, ff, bias, gate, act):
    from krasis_amd import serve_store as S
    cfg = O.make_config(width=width, vocab=70, layers=[O.layer(O.retention(2, 16, 16, [0.9, 0.99]), O.dense(ff)), O.layer(O.attn(2, 1, 16, 0, scale=0.3), O.dense(ff))])
    rng = np.random.default_rng(5)
    W = O.random_weights(cfg, 4)
    for li in range(2):
        for r, n in (("gate", ff), ("up", ff), ("down", width)):
            W[f"l{li}.mlp.{r}.b"] = (0.3 * rng.standard_normal(n)).astype(np.float32)
    W = {k: O.bf16_round(v) for k, v in W.items()}

    def change(spec):
        of = spec.tensors
        for l in spec.layers:
            l.ff_bias = int(bias)
            if act:
                l.dense_act = getattr(S, act)

        def names(s):
            yield from (t for t in of(s) if gate or not t[1].startswith("res_gate"))
            for li in range(2 if bias else 0):
                for r in ("gate", "up", "down"):
                    yield li, r + "_b", 0, f"l{li}.mlp.{r}.b"
        spec.tensors, spec.res_gate = names, int(gate)
    seqs = [tokens(cfg, 5 + r + 4, 40 + r) for r in range(requests)]
    got = []
    for eng in stores(cfg, W, change):
        for r, s in enumerate(seqs):
            eng.step([(r, s[:-4], [])])
        got.append(np.stack([eng.step([(r, [s[i - 4]], [0]) for r, s in enumerate(seqs)])[0] for i in range(4)], 1).astype(np.float64))
    ref, got = got
    e = np.sqrt(((got - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())
    assert np.median(e) < 2e-2 and (e < 4e-2).mean() >= 0.9, e
