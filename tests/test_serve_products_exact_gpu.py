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


# strips: four waves (4096 columns and more) and eight, one block of sixteen rows and two; a wave has 0 - 13 steps of 32 k
@pytest.mark.parametrize("steps", [1, 3, 5, 8, 9, 16, 20, 24, 28, 33, 47, 48, 52, 64, 65, 97])
@pytest.mark.parametrize("want,vocab", [(1, 47), (16, 4097), (32, 33)])
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
