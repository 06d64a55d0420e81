"""The first and the last launch of a serving step: arrays read from pinned host memory, logits and their largest entries stored there.

The rows that come back are compared with the float64 restatement (tolerances of test_serve_gpu.py), the largest entries with the rows themselves, exactly."""
import numpy as np
import pytest

from tests import oracle_serve as O
from tests.test_serve_gpu import engine, rel, tokens

pytestmark = pytest.mark.gpu


def model(vocab, seed, width=64):
    cfg = O.make_config(width=width, vocab=vocab, eps=1e-5, layers=[{"type": "attention", "mixer": O.attn(4, 2, 16, 16, 0, 8, scale=0.25), "mlp": O.dense(24)}])
    return cfg, O.random_weights(cfg, seed)


# vocabularies: fewer entries than one workgroup's, not a multiple of four, one past a workgroup's share, several workgroups; wanted rows: one, one per request, many of a prompt
@pytest.mark.parametrize("vocab", [3, 101, 1025, 4100, 33000])
@pytest.mark.parametrize("dtype,tol", [("float32", 2e-4), ("bfloat16", 4e-2)])
def test_rows_and_largest_entries(vocab, dtype, tol):
    cfg, W = model(vocab, 21)
    a, b = tokens(cfg, 90, 22), tokens(cfg, 40, 23)
    ra, rb = O.forward(cfg, W, a)[0], O.forward(cfg, W, b)[0]
    eng = engine(cfg, W, dtype)
    many = list(range(70)) if vocab < 5000 else list(range(0, 70, 9))
    for entries, ref in (([("a", a[:70], many)], ra[many]),                                             # more tokens than a launch reads itself
                         ([("b", b[:7], [6]), ("a", a[70:74], [0, 3])], np.stack([rb[6], ra[70], ra[73]])),
                         ([("a", [a[74]], [0]), ("b", [b[7]], [0])], np.stack([ra[74], rb[7]])),
                         ([("a", [a[75]], [0])], ra[75:76])):
        logits, amax = eng.step(entries)
        assert rel(logits, ref) < tol
        assert np.array_equal(amax, logits.argmax(-1))
    assert eng.step([("a", [a[76]], []), ("b", [b[8]], [])])[1].size == 0
    logits, amax = eng.step([("a", [a[77]], [0]), ("b", [b[9]], [0])], logits=False)
    assert logits is None
    for r, ref in zip(amax, (ra[77], rb[9])):
        assert ref[r] >= ref.max() - 2 * tol * np.sqrt((ref ** 2).mean())


def test_equal_nan_and_infinite_entries():
    """the lowest index of equal entries (zeros of either sign), a NaN never"""
    cfg, W = model(2000, 24)
    h = np.zeros_like(W["head"])
    for fill, at, want in ((0.0, {}, 0), (-0.0, {7: 0.0}, 0), (0.0, {3: np.nan}, 0), (np.nan, {}, 0), (np.nan, {1500: 0.0}, 1500)):
        h[:] = fill
        for i, v in at.items():
            h[i] = v
        eng = engine(cfg, {**W, "head": h.copy()})
        logits, amax = eng.step([("a", [1], [0])])
        assert amax[0] == want and np.isnan(logits[0]).sum() == np.isnan(h[:, 0]).sum()
    assert engine(cfg, W).step([("a", [1], [0])])[1][0] == O.forward(cfg, W, [1])[0][0].argmax()


# head entries by index, the others at `fill`, and the entry that wins; a step's search is two workgroups' of a thousand entries each here
INF = float("inf")
INFINITE = [(-INF, {}, 0), (-INF, {1500: -2.0}, 1500), (-INF, {3: -2.0, 1999: -3.0}, 3), (np.nan, {1999: -INF}, 1999), (np.nan, {700: -INF, 1700: -INF}, 700),
            (0.5, {1200: INF, 1700: INF}, 1200), (np.nan, {5: INF, 1400: 1.0}, 5), (-1.0, {999: -INF, 1000: INF, 1001: np.nan}, 1000)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_infinite_entries_of_several_rows(dtype):
    """minus infinity wins only where nothing but it and NaN is, plus infinity against everything; three rows a step, in the f32 store and from the bf16 store's strips"""
    cfg, W = model(2000, 25)
    h = np.zeros_like(W["head"])
    h[:64, :64] = np.eye(64)
    step = lambda head: engine(cfg, {**W, "head": head}, dtype).step([(r, [5 + r], [0]) for r in range(3)])
    hidden = step(h)[0][:, :64]                                # the rows that the head multiplies
    col = int(np.argmax(hidden.min(0)))
    assert hidden[:, col].min() > 0.05                         # one column that is positive in all three: a row of logits is that column of the head, scaled
    for fill, at, want in INFINITE:
        h = np.zeros_like(W["head"])
        h[:, col] = fill
        for i, v in at.items():
            h[i, col] = v
        logits, amax = step(h)
        assert (amax == want).all(), (fill, at, amax)
        ref = hidden[:, col:col + 1].astype(np.float64) * h[:, col].astype(np.float64)
        assert np.array_equal(np.isnan(logits), np.isnan(ref)) and np.array_equal(np.isinf(logits), np.isinf(ref)) and np.array_equal(np.sign(logits[np.isinf(logits)]), np.sign(ref[np.isinf(ref)]))
