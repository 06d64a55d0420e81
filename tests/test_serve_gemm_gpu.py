"""The serving store's matrix products at the edges of their forms, against float64.

The vocabulary projection is one product whose three sizes a caller chooses freely -- wanted rows, vocabulary, width -- so it reaches every form of a single matrix: the
strips for few rows (one and two blocks of sixteen rows, four and eight waves), the 64-, 128- and 256-row tiles, and what takes widths that are not whole slots.
The experts of a small mixture reach the grouped forms."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


def stream_model(width, vocab):
    """embedding and head alone: the one layer's attention sees a single key, which stays small"""
    return O.make_config(width=width, vocab=vocab, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 1, 0, scale=0.3), "mlp": None}])


@pytest.mark.parametrize("want,vocab,width", [
    (1, 33, 64), (15, 4097, 96), (16, 4095, 2048), (17, 2559, 128), (31, 47, 160), (32, 2561, 64),            # strips; 32 rows of more than 2560 columns: the small tile
    (33, 129, 64), (63, 257, 192), (64, 255, 128), (65, 64, 96), (127, 511, 320),                            # 64-row tile, and widths of half slots
    (257, 16385, 64), (511, 4224, 128), (2049, 7165, 64), (2304, 7168, 128), (300, 700, 72)])                  # 128- and 256-row tiles with ragged edges; a width of 16-byte pieces only
def test_vocabulary_projection_sizes(want, vocab, width):
    cfg = stream_model(width, vocab); W = O.random_weights(cfg, 11)
    toks = tokens(cfg, want, 12)
    eng = engine(cfg, W, "bfloat16", max_tokens=4096)
    eng.store.set_capture(True)
    logits, amax = eng.step([("a", toks, list(range(want)))])
    x = eng.store.read_capture(want)[-1].astype(np.float64)
    h = O.layer_norm(x, W["final.norm"].astype(np.float64), W["final.norm.b"].astype(np.float64), 1e-5)
    head = W["head"].astype(np.float64)
    ref = h @ head.T
    # the row is rounded to bf16 (half a unit in the last place of eight bits, independent from element to element), the sums are f32
    spread = np.sqrt(((np.abs(h) * 2.0 ** -9) ** 2) @ (head.T ** 2))
    assert np.all(np.abs(logits - ref) <= 6.0 * spread + 1e-5 * np.abs(h) @ np.abs(head.T))
    assert np.array_equal(amax, logits.argmax(-1))


# slots of the operand ring are given back by parts: 1 - 5 slots of 64 k, last tiles of one to four row blocks (256-row tile) and of one and two (128-row tile)
@pytest.mark.parametrize("width", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("want,vocab", [(2050, 7168), (2176, 7168), (2177, 7167), (2300, 7168), (300, 8192), (383, 8191)])
def test_row_blocks_and_slots(want, vocab, width):
    test_vocabulary_projection_sizes(want, vocab, width)


@pytest.mark.parametrize("n", [1, 2, 5, 8, 9, 16, 17, 40, 65, 130, 420])
def test_expert_products_sizes(n):
    # 1 - 840 rows on ten experts: row by row, strips for few rows per expert with the activation inside and outside the launch, 64-row tiles
    cfg = O.make_config(width=128, vocab=61, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 32, 32, 0, 16, scale=0.2), "mlp": O.moe(10, 2, 1, 1, 192, 2.0, 64, 2.0)}])
    W = O.random_weights(cfg, 13); toks = tokens(cfg, n, 14)
    ref_logits, ref_streams = O.forward(cfg, W, toks)
    eng = engine(cfg, W, "bfloat16")
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    d = eng.store.read_capture(n)[0] - ref_streams[0]
    e = np.sqrt((d ** 2).mean(-1)) / np.sqrt((ref_streams[0] ** 2).mean())
    assert (e < 2e-2).mean() >= 0.95          # a row whose second expert was a close call may have taken another one


@pytest.mark.parametrize("mlp,n", [
    (O.dense(481), 1501), (O.dense(1000), 1200), (O.dense(2884), 2305),                                     # behind the layer's other columns: 128-, 128- and 256-column tiles
    (O.moe(3, 3, 1, 1, 264, 1.5), 1700), (O.moe(8, 8, 1, 1, 260, 1.5, 520, 0.8), 2100)])                     # one matrix per expert, and both
def test_activation_from_the_product(mlp, n, width=64):
    # factors that are no whole tiles, with and without whole 16-byte pieces; every expert is chosen, so that no close call hides an error
    cfg = O.make_config(width=width, vocab=61, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 1, 0, scale=0.3), "mlp": mlp}])
    W = O.random_weights(cfg, 15, router_gain=1.0); toks = tokens(cfg, n, 16)
    ref = O.forward(cfg, W, toks)[1][0]
    eng = engine(cfg, W, "bfloat16", max_tokens=4096)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    d = eng.store.read_capture(n)[0] - ref
    # the input row, the two factors' sums and the activation: three independent roundings of 2^-9 each, which the products pass on at their own scale; a lost factor of
    # 260 would alter its rows by 1 / sqrt(260) = 6e-2
    assert np.sqrt((d ** 2).mean(-1)).max() / np.sqrt((ref ** 2).mean()) < 2e-2


@pytest.mark.parametrize("width", [128, 192, 320])                                                             # two, three and five slots of k: the rings by parts behind the pairs
@pytest.mark.parametrize("mlp,n", [(O.dense(1000), 1200), (O.dense(2884), 2305), (O.moe(3, 3, 1, 1, 264, 1.5), 1700)])
def test_activation_from_the_product_of_several_slots(mlp, n, width):
    test_activation_from_the_product(mlp, n, width)


def _clamped_experts(ff, limit=1.5):
    return O, O.make_config(width=64, vocab=61, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 1, 0, scale=0.3), "mlp": O.moe(3, 3, 1, 1, ff, limit)}])


def _biased(ff):
    from tests import oracle_gasavik as G
    return G, G.make_config(width=64, vocab=61, side=0, layers=[G.layer(G.parallel(2, 1, 8, 8, 3, 1, 1, 8, 8), G.dense(ff))])


def _sequential(mlp, *sizes):
    from tests import oracle_ripupel as P
    return P, P.make_config(width=64, vocab=61, layers=[P.layer(P.rglru(64, 1, 2), getattr(P, mlp)(*sizes))])


# the other kinds of activation, and what joins its factors: clamped experts past their limit on the 256-column tile, silu with biases behind the layer's other columns, silu of a
# sequential block (its product begins at the gate columns), silu of experts whose input carries the router's weight.  `wrong`: the model with that part altered
@pytest.mark.parametrize("make,n,wrong", [
    (lambda: _clamped_experts(1000), 2000, lambda m, W: (_clamped_experts(1000, 3.0)[1], W)),
    (lambda: _biased(1001), 1300, lambda m, W: (m, {**W, "l0.mlp.up.b": np.roll(W["l0.mlp.up.b"], 1)})),
    (lambda: _biased(3804), 1500, lambda m, W: (m, {**W, "l0.mlp.gate.b": np.roll(W["l0.mlp.gate.b"], 1)})),
    (lambda: _sequential("dense", 1000), 1200, lambda m, W: (m, {**W, "l0.mlp.up": np.roll(W["l0.mlp.up"], 1, 0)})),
    (lambda: _sequential("moe", 3, 3, 264), 1700, lambda m, W: (m, {**W, "l0.mlp.router": W["l0.mlp.router"][::-1]})),
    (lambda: _sequential("moe", 4, 4, 1000), 2100, lambda m, W: (m, {**W, "l0.mlp.router": W["l0.mlp.router"][::-1]}))])
def test_other_activations_from_the_product(make, n, wrong):
    from tests import test_gasavik_gpu, test_ripupel_gpu
    M, cfg = make()
    W = M.random_weights(cfg, 17, router_gain=1.0) if M is O else {k: M.bf16_round(v) for k, v in M.random_weights(cfg, 17).items()}
    toks = tokens(cfg, n, 18)
    ref = np.asarray(M.forward(cfg, W, toks)[1][0])
    size = np.sqrt((ref ** 2).mean())
    other = wrong(cfg, W)
    few = toks[:40]
    assert np.sqrt(((np.asarray(M.forward(*other, few)[1][0]) - M.forward(cfg, W, few)[1][0]) ** 2).mean(-1)).max() / size > 6e-2
    eng = {O: engine}.get(M) or (test_ripupel_gpu.engine if cfg["architecture"] == "Ripupel" else test_gasavik_gpu.engine)
    eng = eng(cfg, W, "bfloat16", max_tokens=4096)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    # as above: independent roundings of 2^-9 that the products pass on at their own scale
    assert np.sqrt(((eng.store.read_capture(n)[0] - ref) ** 2).mean(-1)).max() / size < 2e-2


@pytest.mark.parametrize("want,vocab,width", [(17, 129, 32), (63, 65, 96), (65, 64, 2048), (130, 257, 64), (1025, 4100, 64), (1024, 4096, 160), (70, 100, 36)])
def test_vocabulary_projection_sizes_f32(want, vocab, width):
    # 64- and 128-row tiles with ragged edges, one slot and many; a width of 16-byte pieces that is no whole slot
    cfg = stream_model(width, vocab); W = O.random_weights(cfg, 17); toks = tokens(cfg, want, 18)
    eng = engine(cfg, W, max_tokens=2048)
    eng.store.set_capture(True)
    logits, amax = eng.step([("a", toks, list(range(want)))])
    h = O.layer_norm(eng.store.read_capture(want)[-1].astype(np.float64), W["final.norm"].astype(np.float64), W["final.norm.b"].astype(np.float64), 1e-5)
    head = W["head"].astype(np.float64)
    # sums of `width` products in f32, the row itself within a few units of its norm
    assert np.all(np.abs(logits - h @ head.T) <= (4.0 + np.sqrt(width)) * 2.0 ** -24 * 2.0 * (np.abs(h) @ np.abs(head.T)))
    assert np.array_equal(amax, logits.argmax(-1))


@pytest.mark.parametrize("n", [9, 40, 130, 700])
def test_expert_products_sizes_f32(n):
    cfg = O.make_config(width=64, vocab=61, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 32, 32, 7, 16, scale=0.2), "mlp": O.moe(5, 5, 1, 1, 96, 2.0, 64, 2.0)}])
    W = O.random_weights(cfg, 19); toks = tokens(cfg, n, 20)
    ref = O.forward(cfg, W, toks)[1][0]
    eng = engine(cfg, W)
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    d = eng.store.read_capture(n)[0] - ref
    assert np.sqrt((d ** 2).mean(-1)).max() / np.sqrt((ref ** 2).mean()) < 2e-5      # f32 sums of at most 128 products, a few in a row


@pytest.mark.parametrize("n,experts", [(1, 2), (1, 3), (2, 4), (3, 4), (4, 4), (5, 2), (8, 2), (9, 2)])
@pytest.mark.parametrize("ff,shared", [(64, 96), (192, 32), (96, 100)])
def test_shared_expert_beside_the_experts(n, experts, ff, shared):
    # up to 16 expert rows both down projections share a launch; a shared width that is no multiple of 32 and an odd number of
    # experts (the factors are not 16-byte aligned then) take their own.  Every expert is chosen: every row counts
    cfg = O.make_config(width=80, vocab=61, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 32, 32, 0, 16, scale=0.2), "mlp": O.moe(experts, experts, 1, 1, ff, 2.0, shared, 2.0)}])
    W = O.random_weights(cfg, 21); toks = tokens(cfg, n, 22)
    ref = O.forward(cfg, W, toks)[1][0]
    eng = engine(cfg, W, "bfloat16")
    eng.store.set_capture(True)
    eng.step([("a", toks, [n - 1])])
    e = np.sqrt(((eng.store.read_capture(n)[0] - ref) ** 2).mean(-1)) / np.sqrt((ref ** 2).mean())
    assert e.max() < 2e-2
