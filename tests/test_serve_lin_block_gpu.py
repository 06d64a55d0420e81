"""Blocks of 64 tokens of the decayed recurrences at the head sizes whose form has no guards (csrc/kr_serve_ops.hip, sv_lin_cout_kernel): 64 and 128 keys, 64 and 128 value columns, and
one size that keeps the guards; the last block of 1 - 64 tokens, waves without tokens, several requests in a step, a second portion on top of the first.
Oracle and bound of an f32 store (2e-4 of the stream's scale): test_midisun_gpu.py."""
import numpy as np
import pytest

from tests import oracle_midisun as O
from tests.test_midisun_gpu import engine, rel, small_model, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 128), (128, 128), (128, 64)])
@pytest.mark.parametrize("kind", ["retention", "mlstm"])
def test_blocks(kind, dim, vdim):
    mixer = O.retention(2, dim, vdim, [0.97, 0.999], base=300.0) if kind == "retention" else O.mlstm(2, dim, vdim, gate_cap=6.0)
    cfg = small_model([O.layer(mixer, None)]); W = O.random_weights(cfg, 81)
    for sizes in ((1, 64, 65), (15, 17, 48), (63, 128, 130), (200,)):
        eng = engine(cfg, W)
        eng.store.set_capture(True)
        seqs = [tokens(cfg, 2 * n, 82 + i) for i, n in enumerate(sizes)]
        for half in (0, 1):
            eng.step([(i, s[half * len(s) // 2:(half + 1) * len(s) // 2], []) for i, s in enumerate(seqs)])
            got = eng.store.read_capture(sum(sizes))[0]
            ref = np.concatenate([O.forward(cfg, W, s)[1][0][half * len(s) // 2:(half + 1) * len(s) // 2] for s in seqs])
            assert rel(got, ref) < 2e-4, (sizes, half)
