"""The serving store's matrix products over whole numbers: every product and every partial sum is one that f32 holds exactly, so the logits are equal to the last bit in any order of sums, and a step of k
that a pipeline loses, takes twice or takes from another row cannot hide in a tolerance.

The stream is the embedding alone (the one layer's output projection is zero), rows of +1 and -1 in equal numbers, whose norm gives them back; norm weights, bias and the vocabulary matrix are small whole
numbers.  The sizes go through the loops of each form: steps of k per wave of the strips (requested four, six and eight together) and their remainders, one to four steps of the f32 rows and what is left of a
step, slots of the operand rings by parts and whole."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, tokens

pytestmark = pytest.mark.gpu


def check(want, vocab, width, dtype):
    cfg = O.make_config(width=width, vocab=vocab, eps=1e-30, layers=[{"type": "attention", "mixer": O.attn(2, 1, 8, 8, 1, 0, scale=0.3), "mlp": None}])
    W = O.random_weights(cfg, 11)
    rng = np.random.default_rng(want * 10007 + vocab * 101 + width)
    W["l0.mix.o"][:] = 0
    W["embed"] = rng.permuted(np.repeat(np.float32([[1, -1]]), width // 2, 1).repeat(vocab, 0), axis=1)
    W["final.norm"] = rng.integers(1, 4, width).astype(np.float32)
    W["final.norm.b"] = rng.integers(-1, 2, width).astype(np.float32)
    W["head"] = rng.integers(-8, 9, (vocab, width)).astype(np.float32)
    toks = tokens(cfg, want, 12)
    eng = engine(cfg, W, dtype, max_tokens=4096)
    logits, amax = eng.step([("a", toks, list(range(want)))])
    ref = (W["embed"][toks] * W["final.norm"] + W["final.norm.b"]).astype(np.float64) @ W["head"].astype(np.float64).T      # below 2^24
    assert np.array_equal(logits, ref), (int((logits != ref).sum()), np.argwhere(logits != ref)[:4].tolist())
    assert np.array_equal(amax, ref.argmax(1))


# strips: four waves (4096 columns and more) and eight, one block of sixteen rows and two, whole lines (up to two rows of these, whose results go to the host) and halves; a wave has 0 - 13 steps of 32 k
@pytest.mark.parametrize("steps", [1, 3, 5, 8, 9, 16, 20, 24, 28, 33, 47, 48, 52, 64, 65, 97])
@pytest.mark.parametrize("want,vocab", [(1, 47), (2, 4097), (16, 4097), (32, 33)])
def test_strips(steps, want, vocab):
    check(want, vocab, 32 * steps, "bfloat16")


# tiles of 64, 128 and 256 rows and columns; one slot of 64 k to nine, last row tiles of one block and of several
@pytest.mark.parametrize("slots", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("want,vocab", [(65, 129), (383, 8191), (300, 8192), (2050, 7168), (2305, 7167)])
def test_tiles(slots, want, vocab):
    check(want, vocab, 64 * slots, "bfloat16")


# a row times a matrix: steps of 256 k four, two and one at a time, a part of a step, widths that are no whole 16-byte pieces
@pytest.mark.parametrize("width", [4, 6, 252, 256, 260, 512, 768, 1022, 1024, 1028, 1280, 1536, 1796, 2048, 2304, 3068])
@pytest.mark.parametrize("want", [1, 2, 4, 8])
def test_f32_rows(width, want):
    check(want, 33, width, "float32")


# 64, 48 and 32 rows a tile; fewer slots of 32 k than the ring has, as many, more
@pytest.mark.parametrize("slots", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("want,vocab", [(17, 129), (63, 127), (129, 4100), (225, 8191)])
def test_f32_tiles(slots, want, vocab):
    check(want, vocab, 32 * slots, "float32")


# ---------------------------------------------------------------------------------------------------------------- decode steps
# First tokens of T requests: attention's one key has all the weight, so the mixer's output is its values.  Column 0 of every token's embedding is +1, and gates have 64 times it: their
# sigmoid is one to the last bit.  Products of gates and factors are whole numbers that are rounded to bf16 once; experts' weights are 1 or 1 / 2.  So the streams are equal to the last bit.
def embedding(rng, tokens, width, code=None):
    """[tokens, width] of +1 and -1 in equal numbers, +1 in column 0, -1 in column 1, then (code) their bits and the bits' complements"""
    head = np.ones((tokens, 2), np.float32); head[:, 1] = -1
    if code is not None:
        bits = 2.0 * ((code[:, None] >> np.arange(8)) & 1) - 1
        head = np.concatenate([head, bits, -bits], 1).astype(np.float32)
    rest = width - head.shape[1]
    return np.concatenate([head, rng.permuted(np.repeat(np.float32([[1, -1]]), rest // 2, 1).repeat(tokens, 0), axis=1)], 1)


def sparse(rng, rows, cols, n, gate=False):
    """[rows, cols] with n entries of +1 or -1 a row (fewer where they meet), all over the columns; gate: 64 in column 0"""
    w = np.zeros((rows, cols), np.float32)
    w[np.arange(rows)[:, None], rng.integers(0, cols, (rows, n))] = rng.choice(np.float32([-1, 1]), (rows, n))
    if gate:
        w[:, 0] = 64
    return w


def streams(eng, vocab):
    eng.store.set_capture(True)
    eng.step([(t, [t], [0]) for t in range(vocab)])
    return eng.store.read_capture(vocab)[-1]


# a wave's steps of 32 k: none, one, odd and even numbers of them, several rounds of eight.  Rows of the experts: each alone (up to 24, among them rows that share an expert) and in strips,
# down projections of up to sixteen and of more rows, one to sixteen rows an expert
@pytest.mark.parametrize("width,heads,ff,shared_ff", [(96, 1, 32, 32), (352, 2, 160, 96), (1088, 3, 544, 224), (2080, 9, 992, 768)])
@pytest.mark.parametrize("T,top,experts", [(1, 1, 4), (2, 2, 8), (3, 2, 4), (12, 2, 16), (13, 2, 8), (16, 1, 2), (16, 2, 8), (16, 2, 64)])
def test_joined_decode_step(T, top, experts, width, heads, ff, shared_ff):
    cfg = O.make_config(width=width, vocab=T, eps=1e-30, layers=[{"type": "attention", "mixer": O.attn(heads, 1, 32, 32, 0, 0, scale=0.3), "mlp": O.moe(experts, top, 1, 1, ff, 4096.0, shared_ff, 4096.0)}])
    W = O.random_weights(cfg, 11)
    rng = np.random.default_rng(T * 10007 + experts * 101 + width)
    choice = rng.integers(0, experts // top, T)                     # of expert `choice`, or of the pair with that number
    W["embed"] = x = embedding(rng, T, width, choice)
    W["l0.norm1"], W["l0.norm1.b"] = np.ones(width, np.float32), np.zeros(width, np.float32)
    W["l0.mix.sink"][:] = -1000
    W["l0.mix.v"], W["l0.mix.o"] = sparse(rng, 32, width, 20), sparse(rng, width, heads * 32, 20)
    of = np.arange(experts) // top
    W["l0.mlp.router"][:] = 0
    W["l0.mlp.router"][:, 2:10] = 128.0 * (2.0 * ((of[:, None] >> np.arange(8)) & 1) - 1)
    for name, F in [(f"e{e}", ff) for e in range(experts)] + [("shared", shared_ff)]:
        W[f"l0.mlp.{name}.gate"], W[f"l0.mlp.{name}.up"], W[f"l0.mlp.{name}.down"] = sparse(rng, F, width, 24, True), sparse(rng, F, width, 24), sparse(rng, width, F, 24)
    want = x + np.tile(x @ W["l0.mix.v"].T, (1, heads)) @ W["l0.mix.o"].T

    def feed_forward(h, name):
        g, u = h @ W[f"l0.mlp.{name}.gate"].T, h @ W[f"l0.mlp.{name}.up"].T
        assert g.min() >= 16
        return O.bf16_round(g * (u + 1)) @ W[f"l0.mlp.{name}.down"].T
    want = want + feed_forward(x, "shared")
    for t in range(T):
        want[t] += sum(feed_forward(x[t:t + 1], f"e{top * choice[t] + j}")[0] for j in range(top)) / top
    got = streams(engine(cfg, W, "bfloat16", max_tokens=4096, max_slots=T), T)
    assert np.array_equal(got, want), (int((got != want).sum()), np.argwhere(got != want)[:4].tolist())


# a sequential block: mixer projections beside the residual gate's, then gate and up as pairs with the other gate's product behind them
@pytest.mark.parametrize("width,heads,ff", [(96, 1, 32), (352, 2, 160), (1088, 3, 544), (2080, 9, 4128)])
@pytest.mark.parametrize("T", [1, 2, 3, 15, 16])
def test_strips_of_a_sequential_step(T, width, heads, ff):
    from tests import oracle_midisun as M
    from tests.test_midisun_gpu import engine as midisun
    rng = np.random.default_rng(T * 101 + width)
    x = embedding(rng, T, width)
    for part in ("mixer", "feed-forward"):
        cfg = M.make_config(width, T, [M.layer(M.attn(heads, 1, 32, 0, scale=0.3), M.dense(ff) if part == "feed-forward" else None)], eps=1e-30, groups=1, embed_scale=1.0)
        W = M.random_weights(cfg, 11)
        W["embed"] = x
        for name in W:
            leaf = name.split(".")[-1]
            if leaf in ("norm1", "norm2"):
                W[name][:] = 1
            if leaf == "canon1" or leaf == "b":
                W[name][:] = 0
            if leaf in ("rg1", "rg2"):
                W[name] = sparse(rng, width, width, 24, True)
        W["l0.mix.sink"][:] = -1000
        W["l0.mix.k"], W["l0.mix.g"] = sparse(rng, 32, width, 20), sparse(rng, heads, width, 20, True)
        if part == "mixer":
            W["l0.mix.o"] = sparse(rng, width, heads * 32, 20)
            want = x + np.tile(x @ W["l0.mix.k"].T, (1, heads)) @ W["l0.mix.o"].T
        else:
            W["l0.mix.o"][:] = 0
            W["l0.mlp.gate"], W["l0.mlp.up"], W["l0.mlp.down"] = sparse(rng, ff, width, 24, True), sparse(rng, ff, width, 24), sparse(rng, width, ff, 24)
            want = x + O.bf16_round((x @ W["l0.mlp.gate"].T) * (x @ W["l0.mlp.up"].T)) @ W["l0.mlp.down"].T
        got = streams(midisun(cfg, W, "bfloat16", max_tokens=4096, max_slots=T), T)
        assert np.array_equal(got, want), (part, int((got != want).sum()), np.argwhere(got != want)[:4].tolist())
