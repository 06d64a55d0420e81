"""The 128-row attention of prompt portions (bf16 store) at the edges of its tiles, against the float64 restatement: head sizes and groupings it is compiled for, portions around the
tile sizes, windows around the key tile, portions deep in a request whose keys are shared over several workgroups, unequal requests in one step."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


def model(heads, kv_heads, dim, vdim, window, rot=0):
    return O.make_config(width=128, vocab=50, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(heads, kv_heads, dim, vdim, window, rot, scale=2.0 * dim ** -0.5), "mlp": None}])


def row_errors(got, ref):
    """error of every row, relative to the root mean square of the layer's own contribution over the rows"""
    return np.sqrt(((got - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 4, 32, 32), (2, 1, 32, 128), (8, 2, 64, 64), (16, 1, 64, 32), (32, 1, 32, 64), (8, 1, 128, 128), (4, 2, 128, 64), (2, 2, 64, 128), (16, 2, 128, 32)])
@pytest.mark.parametrize("n,window", [(32, 0), (33, 7), (65, 64), (129, 65), (200, 1), (257, 130)])
def test_portion_sizes(heads, kv_heads, dim, vdim, n, window):
    cfg = model(heads, kv_heads, dim, vdim, window, rot=16); W = O.random_weights(cfg, 21)
    toks = tokens(cfg, n, 22)
    eng = engine(cfg, W, "bfloat16")
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    got = eng.store.read_capture(n)[0]
    ref = O.forward(cfg, W, toks)[1][0]
    x0 = W["embed"].astype(np.float64)[np.asarray(toks)]
    # bf16 holds the normed input, keys, values and the mixed rows: four roundings of 2^-9 a value, averaged over the row
    assert row_errors(got - x0, ref - x0).max() < 2e-2


@pytest.mark.parametrize("window", [0, 700])
def test_portions_deep_in_a_request_share_keys(window):
    # 1500 tokens in the cache, then 40 and 33 more of two requests and one token of a third in one step: the keys of every tile go over several workgroups
    cfg = model(8, 2, 64, 64, window); W = O.random_weights(cfg, 23)
    a, b, c = tokens(cfg, 1540, 24), tokens(cfg, 1300, 25), tokens(cfg, 90, 26)
    eng = engine(cfg, W, "bfloat16", max_tokens=8192)
    for rid, t, k in (("a", a, 1500), ("b", b, 1267), ("c", c, 89)):
        eng.step([(rid, t[:k], [])])
    eng.store.set_capture(True)
    eng.step([("c", c[89:], [0]), ("a", a[1500:], [39]), ("b", b[1267:], [32])])
    got = eng.store.read_capture(74)[0]
    lo = 0
    for t, k in ((c, 89), (a, 1500), (b, 1267)):
        n = len(t) - k
        ref = O.forward(cfg, W, t)[1][0][k:]
        x0 = W["embed"].astype(np.float64)[np.asarray(t[k:])]
        assert row_errors(got[lo:lo + n] - x0, ref - x0).max() < 2e-2
        lo += n


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(6, 3, 32, 64), (5, 1, 64, 32), (16, 1, 64, 128), (40, 1, 32, 32), (8, 2, 128, 128)])
@pytest.mark.parametrize("ctx,window", [(1, 0), (31, 3), (64, 33), (255, 0), (700, 0), (1300, 290)])
def test_single_tokens(heads, kv_heads, dim, vdim, ctx, window):
    # three requests, one token each, at positions around the 32-key tile, inside one workgroup and split over several; groups of 2 - 40 heads per key head
    cfg = model(heads, kv_heads, dim, vdim, window, rot=8); W = O.random_weights(cfg, 27)
    seqs = [tokens(cfg, n + 1, 28 + i) for i, n in enumerate((ctx, max(1, ctx - 5), max(1, ctx // 2)))]
    eng = engine(cfg, W, "bfloat16", max_tokens=8192)
    for i, s in enumerate(seqs):
        eng.step([(i, s[:-1], [])])
    eng.store.set_capture(True)
    eng.step([(i, s[-1:], [0]) for i, s in enumerate(seqs)])
    got = eng.store.read_capture(3)[0]
    x0 = W["embed"].astype(np.float64)[[s[-1] for s in seqs]]
    ref = np.stack([O.forward(cfg, W, s)[1][0][-1] for s in seqs])
    assert row_errors(got - x0, ref - x0).max() < 2e-2


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,keep,window", [
    (4, 2, 32, 32, 1, 12), (4, 1, 64, 128, 4, 64), (4, 4, 128, 64, 31, 33), (8, 2, 32, 64, 33, 31), (4, 1, 128, 128, 40, 40), (4, 2, 64, 32, 3, 12),
    (4, 2, 64, 64, 4, 290), (4, 1, 128, 128, 33, 290), (8, 2, 32, 32, 40, 250)])                 # the last ones share their keys over several workgroups
def test_kept_first_keys_meet_the_window(heads, kv_heads, dim, vdim, keep, window):
    # every position from the one where the window still touches the kept keys to one where a block of 32 keys lies between them: a kept key counts once
    from tests import oracle_gasavik as G
    from tests.test_gasavik_gpu import engine as gasavik_engine
    cfg = G.make_config(width=64, vocab=50, side=0, layers=[G.layer(G.parallel(heads, kv_heads, dim, vdim, window, keep, 1, 8, 8, left_scale=1.0, right_scale=0.01), None)])
    W = {k: G.bf16_round(v) for k, v in G.random_weights(cfg, 29).items()}
    first, n = keep + window - 1, keep + window + 62
    toks = tokens(cfg, n, 30)
    eng = gasavik_engine(cfg, W, "bfloat16")
    eng.step([("a", toks[:first], [])])
    eng.store.set_capture(True)
    got = []
    for i in range(first, first + 42):
        eng.step([("a", toks[i:i + 1], [0])])
        got.append(eng.store.read_capture(1)[0])
    eng.step([("a", toks[first + 42:], [0])])                                                        # a portion short of the prompt form
    got = np.concatenate(got + [eng.store.read_capture(n - first - 42)[0]])
    x0 = G.embed(cfg, {k: np.asarray(v, np.float64) for k, v in W.items()}, toks)[first:]
    # as above; one key of 291 twice would be off by 1 / sqrt(291) = 6e-2
    assert row_errors(got - x0, G.forward(cfg, W, toks)[1][0][first:] - x0).max() < 2e-2


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,requests", [(8, 8, 32, 64, 24), (8, 2, 64, 32, 40), (16, 1, 128, 128, 33)])
def test_many_requests_deep_in_their_caches(heads, kv_heads, dim, vdim, requests):
    # more workgroups than the chip holds: fewer shares each.  Every request is the beginning of one sequence, so one row of the oracle each
    cfg = model(heads, kv_heads, dim, vdim, 0, rot=8); W = O.random_weights(cfg, 31)
    toks = tokens(cfg, 1060 + requests, 32)
    eng = engine(cfg, W, "bfloat16", max_tokens=requests * 1152, max_slots=requests)
    for i in range(requests):
        eng.step([(i, toks[:1060 + i], [])])
    eng.store.set_capture(True)
    eng.step([(i, toks[1060 + i:1061 + i], [0]) for i in range(requests)])
    got = eng.store.read_capture(requests)[0]
    x0 = W["embed"].astype(np.float64)[toks[1060:1060 + requests]]
    assert row_errors(got - x0, O.forward(cfg, W, toks)[1][0][1060:] - x0).max() < 2e-2


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(8, 2, 64, 64), (16, 1, 64, 128), (4, 4, 128, 32)])
@pytest.mark.parametrize("portion", [33, 260])
def test_short_entries_beside_a_portion(heads, kv_heads, dim, vdim, portion):
    # a portion at the start of a request beside single tokens and a few tokens deep in others: the short entries take launches of their own, in any order of the entries
    cfg = model(heads, kv_heads, dim, vdim, 0); W = O.random_weights(cfg, 33)
    a, b, c = tokens(cfg, 1500, 34), tokens(cfg, portion, 35), tokens(cfg, 40, 36)
    x0, ref = [W["embed"].astype(np.float64)[np.asarray(t)] for t in (a, b, c)], [O.forward(cfg, W, t)[1][0] for t in (a, b, c)]
    eng = engine(cfg, W, "bfloat16", max_tokens=8192, max_slots=6)
    for rid, n in (("a", 1495), ("b", 1300), ("d", 1409)):                 # beginnings of one sequence
        eng.step([(rid, a[:n], [])])
    eng.store.set_capture(True)
    eng.step([("d", a[1409:1410], [0]), ("p", b, [portion - 1]), ("a", a[1495:], [4]), ("q", c, [39]), ("b", a[1300:1301], [0])])
    got = eng.store.read_capture(portion + 47)[0]
    lo = 0
    for i, k, n in ((0, 1409, 1), (1, 0, portion), (0, 1495, 5), (2, 0, 40), (0, 1300, 1)):
        assert row_errors(got[lo:lo + n] - x0[i][k:k + n], ref[i][k:k + n] - x0[i][k:k + n]).max() < 2e-2
        lo += n


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(8, 8, 32, 64), (16, 2, 128, 128), (32, 1, 64, 32)])
@pytest.mark.parametrize("n", [2, 7, 31])
def test_many_short_portions(heads, kv_heads, dim, vdim, n):
    cfg = model(heads, kv_heads, dim, vdim, 0, rot=8); W = O.random_weights(cfg, 37)
    requests = 1 + 192 // (n * kv_heads * max(1, heads // kv_heads // 16))
    toks = tokens(cfg, 70 + requests + n, 38)
    eng = engine(cfg, W, "bfloat16", max_tokens=requests * 320, max_slots=requests)
    for i in range(requests):
        eng.step([(i, toks[:70 + i], [])])
    eng.store.set_capture(True)
    eng.step([(i, toks[70 + i:70 + i + n], [0]) for i in range(requests)])
    got = eng.store.read_capture(requests * n)[0]
    at = np.concatenate([np.arange(70 + i, 70 + i + n) for i in range(requests)])
    x0 = W["embed"].astype(np.float64)[np.asarray(toks)[at]]
    assert row_errors(got - x0, O.forward(cfg, W, toks)[1][0][at] - x0).max() < 2e-2


@pytest.mark.parametrize("design,size", [("capped", 4096), ("capped", 330), ("chunked", 0), ("chunked", 300)])
@pytest.mark.parametrize("heads,kv_heads,dim", [(8, 2, 128), (16, 4, 64)])
def test_capped_scores_distance_bias_and_chunks(design, size, heads, kv_heads, dim):
    # a prompt of 700 tokens as portions of 40 and 660 (one and several workgroups per token's keys), 6 tokens at once, then single ones; a soft cap near the scores' size
    from tests import oracle_midisun as M, oracle_pamulix as P, test_midisun_gpu, test_pamulix_gpu
    if design == "capped":
        cfg = M.make_config(64, 50, [M.layer(M.attn(heads, kv_heads, dim, size, scale=0.2, softcap=2.5), None)], groups=1, taps=1)
        W = {k: M.bf16_round(v) for k, v in M.random_weights(cfg, 39).items()}
        make, forward, x0 = test_midisun_gpu.engine, M.forward, lambda t: W["embed"].astype(np.float64)[t] * cfg["embedding"]["scale"]
    else:
        cfg = P.make_config(width=64, vocab=50, layers=[P.layer(P.attn(heads, kv_heads, dim, dim, size, scale=0.2), None)])
        W = P.random_weights(cfg, 39)
        make, forward, x0 = test_pamulix_gpu.engine, P.forward, lambda t: W["embed"].astype(np.float64)[t]
    toks = tokens(cfg, 716, 40)
    eng = make(cfg, W, "bfloat16")
    eng.store.set_capture(True)
    got, at = [], 0
    for n in [40, 660, 6] + [1] * 10:
        eng.step([("a", toks[at:at + n], [n - 1])])
        got.append(eng.store.read_capture(n)[0])
        at += n
    base = x0(np.asarray(toks))
    assert row_errors(np.concatenate(got) - base, forward(cfg, W, toks)[1][0] - base).max() < 2e-2


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(16, 2, 128, 128), (4, 4, 128, 64), (32, 1, 128, 256)])
@pytest.mark.parametrize("ctx,window", [(15, 0), (16, 7), (63, 0), (64, 17), (65, 0), (300, 130), (700, 0)])
def test_single_tokens_f32(heads, kv_heads, dim, vdim, ctx, window):
    # blocks of 16 keys a wave, one workgroup and several; a step of 130 single tokens, past the line, takes 64 again
    cfg = model(heads, kv_heads, dim, vdim, window, rot=8); W = O.random_weights(cfg, 61)
    for requests in (2, 130 if ctx == 65 else 1):
        seqs = [tokens(cfg, max(1, ctx - i % 3) + 1, 62 + i % 3) for i in range(requests)]
        eng = engine(cfg, W, max_tokens=2048 + 128 * requests, max_slots=requests)
        for i, s in enumerate(seqs):
            eng.step([(i, s[:-1], [])])
        eng.store.set_capture(True)
        eng.step([(i, s[-1:], [0]) for i, s in enumerate(seqs)])
        got = eng.store.read_capture(requests)[0]
        x0 = W["embed"].astype(np.float64)[[s[-1] for s in seqs]]
        kinds = [O.forward(cfg, W, s)[1][0][-1] for s in seqs[:3]]
        ref = np.stack([kinds[i % 3] for i in range(requests)])
        assert row_errors(got - x0, ref - x0).max() < 2e-5      # f32 throughout: sums of some hundred products and exponentials, each within 2^-23
