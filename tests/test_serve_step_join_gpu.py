"""Decode steps of a parallel block with experts in a bf16 store, where attention and the experts share launches (csrc/kr_serve_step.hip), against the float64 restatement.

The sizes are the edges of those launches: rows that are each taken alone (up to 24) and the next one, strips and columns that do not fill a workgroup, up to sixteen tokens, one
and several shares of a token's keys, one and two batches of sixteen query heads, more than 64 experts.  Tolerance: that of the store's other bf16 tests (test_serve_gpu.py)."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,mixer,mlp,requests,length,steps", [
    ("one_row_shares_of_keys", O.attn(8, 2, 32, 64, 0, 16, base=100.0, scale=0.2), O.moe(4, 1, 1, 1, 32, 1.5), 1, 600, 6),
    ("24_rows", O.attn(8, 4, 64, 32, 0, 32, scale=0.15), O.moe(16, 3, 4, 2, 32, 1.5, 96, 2.0), 8, 30, 4),
    ("25_rows", O.attn(8, 4, 64, 32, 19, 32, scale=0.15), O.moe(16, 5, 1, 1, 32, 1.5, 96, 2.0), 5, 30, 4),
    ("sixteen_tokens_many_experts", O.attn(16, 1, 128, 128, 70, 64, scale=0.09), O.moe(128, 8, 1, 1, 160, 1.2, 64, 1.0), 16, 40, 3),
    ("sixteen_tokens_few_experts", O.attn(2, 2, 128, 64, 0, 0, scale=0.09), O.moe(4, 2, 1, 1, 96, 1.2), 16, 20, 3),
    ("two_batches_of_heads", O.attn(32, 1, 64, 64, 0, 64, scale=0.12), O.moe(8, 2, 2, 1, 64, 1.5, 64, 2.0), 3, 300, 3),
])
def test_steps_close_to_oracle(name, mixer, mlp, requests, length, steps):
    cfg = O.make_config(width=160, vocab=90, eps=1e-5, layers=[{"type": "attention", "mixer": mixer, "mlp": mlp}] * 2)
    W = O.random_weights(cfg, 11)
    lens = [length - (3 * r) % max(1, length // 2) for r in range(requests)]
    seqs = [tokens(cfg, n + steps, 100 + r) for r, n in enumerate(lens)]
    eng = engine(cfg, W, "bfloat16", max_tokens=64 * requests * ((length + steps) // 64 + 1), max_slots=requests)
    eng.step([(r, s[:n], []) for r, (s, n) in enumerate(zip(seqs, lens))])
    got = np.stack([eng.step([(r, [s[n + i]], [0]) for r, (s, n) in enumerate(zip(seqs, lens))])[0] for i in range(steps)], 1)
    ref = np.stack([O.forward(cfg, W, s)[0][n:] for s, n in zip(seqs, lens)])
    e = np.sqrt(((got - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())
    assert np.median(e) < 2e-2 and (e < 4e-2).mean() >= 0.9, (name, e)


@pytest.mark.parametrize("ff", [1024, 4096])
def test_more_rows_than_experts(ff):
    """each row alone while the experts' matrices stay in the cache, strips beyond (five experts of 2 x 4096 x 2048 are 168 MB); against the f32 store, which other tests hold to the
    float64 restatement"""
    cfg = O.make_config(width=2048, vocab=50, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 64, 64, 0, 0, scale=0.12), "mlp": O.moe(5, 2, 1, 1, ff, 1.5)}])
    W = O.random_weights(cfg, 15)
    seqs = [tokens(cfg, 8, 60 + r) for r in range(6)]
    got = []
    for dtype in ("float32", "bfloat16"):
        eng = engine(cfg, W, dtype, max_slots=6)
        eng.step([(r, s[:5], []) for r, s in enumerate(seqs)])
        got.append(np.stack([eng.step([(r, [s[5 + i]], [0]) for r, s in enumerate(seqs)])[0] for i in range(3)], 1).astype(np.float64))
    e = np.sqrt(((got[1] - got[0]) ** 2).mean(-1)) / np.sqrt((got[0] ** 2).mean())
    assert np.median(e) < 2e-2 and (e < 4e-2).mean() >= 0.9, e


def test_a_step_is_the_same_every_time_and_under_replay():
    """joined launches leave the same bits eagerly and from a replayed graph, whatever ran in between"""
    cfg = O.make_config(width=128, vocab=70, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(8, 2, 128, 128, 0, 64, scale=0.1), "mlp": O.moe(8, 3, 1, 1, 96, 1.5, 64, 2.0)}] * 2)
    W = O.random_weights(cfg, 12)
    a, b = tokens(cfg, 330, 13), tokens(cfg, 330, 14)
    runs = []
    for graph in (True, False):
        eng = engine(cfg, W, "bfloat16")
        eng.store.set_use_graph(graph)
        eng.step([("a", a[:240], []), ("b", b[:9], [])])
        runs.append([eng.step([("a", [a[240 + i]], [0]), ("b", [b[9 + i]], [0])])[0] for i in range(40)])       # past 256 keys: another share count on the way
        assert (eng.store.graph_replays() > 0) == graph
    assert all(np.array_equal(x, y) for x, y in zip(*runs))


# what a joined layer may have beside the plain design; the second layer of two, where it refers to the first
OPTIONS = {
    "gate_per_head": dict(out_gate="OGATE_HEAD_SIGMOID"), "gate_per_element": dict(out_gate="OGATE_ELEM_SIGMOID"), "values_mixed": dict(v_mix="VMIX_BLEND"),
    "convolution": dict(proj_conv=3), "norm_of_whole_rows": dict(qk_unit_norm="QKNORM_WHOLE"), "norm_with_weight": dict(qk_unit_norm="QKNORM_WEIGHTED"), "soft_cap": dict(softcap=1.5),
    "distance": dict(dist_bias=1), "kept_keys": dict(window=12, keep_first=3), "kept_keys_past_a_tile": dict(window=5, keep_first=33), "chunk": dict(chunk=16), "sink": dict(has_sink="SINK_ZERO"),
    "weights_on_inputs": dict(expert_in_weight=1), "keys_of_another_layer": dict(kv_from=0), "values_are_keys": dict(v_from_k=1), "biases": dict(proj_bias=2),
}


@pytest.mark.parametrize("name", OPTIONS)
def test_every_mechanism_of_a_joined_layer(name):
    """tokens one by one, each step joined, against the same tokens as one prompt, whose launches are not; the prompt's own distance to 64 bits is other tests' matter.  Tolerance: as above"""
    from krasis_amd import serve_store as S
    o = {k: getattr(S, v) if isinstance(v, str) else v for k, v in OPTIONS[name].items()}
    base = dict(heads=4, kv_heads=2, dim=32, vdim=32, rot_dims=16, scale=0.18, mlp_kind=S.MLP_MOE, experts=6, top=2, expert_ff=64, expert_act=S.ACT_SILU, shared_ff=32)
    first = {**base, **({"v_mix": S.VMIX_FIRST} if "v_mix" in o else {} if "kv_from" in o else o)}
    store = S.ServeStore(80, 64, [S.LayerSpec(**first), S.LayerSpec(**{**base, **o})], max_slots=4, pool_tokens=1024)
    store.fill_synthetic(seed=41, amp=2.5)
    store.finalize()
    rng = np.random.default_rng(42)
    seqs = [rng.integers(0, 80, n) for n in (70, 61, 50)]
    ref, slots = [], [store.admit() for _ in seqs]
    for sl, s in zip(slots, seqs):
        ref.append(store.step([(sl, s)], range(len(s) - 20, len(s)))[0])
        store.release(sl)
    slots = [store.admit() for _ in seqs]
    for sl, s in zip(slots, seqs):
        store.step([(sl, s[:-20])], [])
    got = np.stack([store.step([(sl, [s[len(s) - 20 + i]]) for sl, s in zip(slots, seqs)], range(3))[0] for i in range(19)], 1).astype(np.float64)
    store.set_profiling(True)
    last = store.step([(sl, [s[-1]]) for sl, s in zip(slots, seqs)], range(3))[0]
    assert store.profile()[3] == 0                              # attention had no launch of its own
    store.set_profiling(False)
    got, ref = np.concatenate([got, last[:, None]], 1), np.stack(ref).astype(np.float64)
    e = np.sqrt(((got - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())
    assert np.median(e) < 2e-2 and (e < 4e-2).mean() >= 0.9, (name, e)


@pytest.mark.parametrize("requests", [2, 12])
@pytest.mark.parametrize("ff", [96, 384, 640, 768, 1024, 1408])
def test_steps_of_k_requested_together(ff, requests):
    """a wave's share of the down projections is 1, 3, 5, 6, 8 and 11 steps of 32 k, requested four, six or eight at a time, beside attention's projection six or eight at a time (few and
    many expert rows); the prompts' fifteen and sixty rows meet the same strips in launches of their own"""
    cfg = O.make_config(width=256, vocab=50, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 64, 64, 0, 0, scale=0.12), "mlp": O.moe(10, 2, 1, 1, ff, 1.5, ff, 1.5)}])
    W = O.random_weights(cfg, 21)
    seqs = [tokens(cfg, 8, 70 + r) for r in range(requests)]
    eng = engine(cfg, W, "bfloat16", max_slots=requests)
    first = eng.step([(r, s[:5], [4]) for r, s in enumerate(seqs)])[0]
    got = np.stack([first] + [eng.step([(r, [s[5 + i]], [0]) for r, s in enumerate(seqs)])[0] for i in range(3)], 1)
    ref = np.stack([O.forward(cfg, W, s)[0][4:] for s in seqs])
    e = np.sqrt(((got - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())
    assert np.median(e) < 2e-2 and (e < 4e-2).mean() >= 0.9, (ff, requests, e)
