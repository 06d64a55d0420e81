"""The exact grouped GEMM for many rows against the 64-row tiles, bit for bit: the same tokens in one call and in calls of forty rows, which take the latter.  An odd number of quantization groups,
columns that are no whole tile, experts of 1, 63 - 65 and 127 - 129 rows, skipped slots, and a shared expert of 128 and more tiles."""
import numpy as np
import pytest

from tests.test_prefill_gpu import _setup
from tests.test_prefill_strips_gpu import _cut
from tests.util import rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,bits,w2_bits,n_shared", [(640, 384, 4, 4, 1), (384, 256, 8, 8, 1), (640, 128, 4, 8, 0), (256, 640, 8, 4, 0)])
def test_many_rows_equal_few(H, I, bits, w2_bits, n_shared):
    E, k = 9, 2
    eng, mgr, experts, shared, rng, torch = _setup(H, I, E, k, n_shared, 1.5 if n_shared else 1.0, bits=bits, w2_bits=w2_bits)
    M = 7000 if n_shared else 700
    x = torch.from_numpy(rand_bf16(rng, (M, H)).view(np.int16)).cuda().view(torch.bfloat16)
    ids = np.full((M, k), -1, np.int32)
    ids[:, 0] = 8
    at = 0
    for e, n in enumerate((1, 63, 64, 65, 127, 128, 129, 0)):
        ids[at:at + n, 1] = e; at += n
    ids[at] = -1                                                     # a token without experts
    ids = torch.from_numpy(ids).cuda(); w = torch.from_numpy(rng.random((M, k)).astype(np.float32)).cuda()
    whole = mgr.forward(0, x, ids, w).view(torch.int16).cpu().numpy()
    few = np.concatenate([mgr.forward(0, x[i:i + 40], ids[i:i + 40], w[i:i + 40]).view(torch.int16).cpu().numpy() for i in range(0, M, 40)])
    assert np.array_equal(whole, few)


@pytest.mark.parametrize("M", [216, 256, 257, 601])
@pytest.mark.parametrize("H,I,bits,w2_bits,n_shared", [(640, 384, 4, 4, 1), (384, 256, 8, 8, 2), (256, 640, 8, 4, 1), (256, 128, 4, 8, 2)])
def test_shared_expert_in_the_experts_launches(M, H, I, bits, w2_bits, n_shared):
    # fewer shared tiles than a launch of its own would take, whole and ragged row tiles, matrices of either type; forty rows at a time take neither the wide kernel nor the join
    E, k = 9, 2
    eng, mgr, experts, shared, rng, torch = _setup(H, I, E, k, n_shared, 1.5, bits=bits, w2_bits=w2_bits)
    x = torch.from_numpy(rand_bf16(rng, (M, H)).view(np.int16)).cuda().view(torch.bfloat16)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(M)]).astype(np.int32); ids[5] = -1
    ids = torch.from_numpy(ids).cuda(); w = torch.from_numpy(rng.random((M, k)).astype(np.float32)).cuda()
    whole = mgr.forward(0, x, ids, w).view(torch.int16).cpu().numpy()
    few = np.concatenate([mgr.forward(0, x[i:i + 40], ids[i:i + 40], w[i:i + 40]).view(torch.int16).cpu().numpy() for i in range(0, M, 40)])
    assert np.array_equal(whole, few)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("limit", [0.0, 0.75])
def test_hidden_digits_of_the_gate_and_up_launch(bits, limit):
    # the wide kernel's own digits against the activation's launch (forty rows at a time), both activations: rows of exact zeros (a scale of one), a row far past the clamp, ragged tiles
    import torch
    from krasis_amd import GpuPrefillManager, KrasisEngine, ModelConfig
    from tests.util import make_experts, upload
    H, I, E, k, M = 384, 384, 5, 2, 301
    rng = np.random.default_rng(7)
    experts, shared = make_experts(rng, E, H, I, bits), make_experts(rng, 1, H, I, bits)[0]
    eng = KrasisEngine(); eng.configure(ModelConfig(H, I, E, k, 1, 1, 1.0, swiglu_limit=limit, activation_alpha=1.702))
    upload(eng, 0, experts, shared)
    mgr = GpuPrefillManager(eng, k)
    x = rand_bf16(rng, (M, H)); x[3] = 0; x[200] = 0
    x = torch.from_numpy(x.view(np.int16)).cuda().view(torch.bfloat16)
    x[17] *= 64
    ids = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(M)]).astype(np.int32)).cuda(); w = torch.from_numpy(rng.random((M, k)).astype(np.float32)).cuda()
    counts = np.bincount(ids.flatten().cpu().numpy(), minlength=E)
    whole = mgr.forward(0, x, ids, w).view(torch.int16).cpu().numpy()
    assert _cut(eng) == (sum(-(-c // 128) for c in counts), 0) and _cut(eng)[0] < sum(-(-c // 64) for c in counts)      # the wide kernel's tiles
    few = []
    for i in range(0, M, 40):
        few.append(mgr.forward(0, x[i:i + 40], ids[i:i + 40], w[i:i + 40]).view(torch.int16).cpu().numpy())
        counts = np.bincount(ids[i:i + 40].flatten().cpu().numpy(), minlength=E)
        assert _cut(eng) in ((sum(-(-c // 64) for c in counts), 0), (0, sum(-(-c // 32) for c in counts)), (0, sum(-(-c // 16) for c in counts)))
    assert np.array_equal(whole, np.concatenate(few)) and np.any(whole[17]) and not np.any(whole[3] & 0x7FFF)


def test_gate_and_up_take_no_memory():
    """2400 rows whose hidden digits leave the first launch: 39 MB of gate and up in f32 are not kept, only what a pass of fewer rows may leave"""
    E, k, M, H, I = 9, 2, 1200, 256, 2048
    eng, mgr, experts, shared, rng, torch = _setup(H, I, E, k, 1, 1.0)
    x = torch.from_numpy(rand_bf16(rng, (M, H)).view(np.int16)).cuda().view(torch.bfloat16)
    ids = torch.from_numpy(np.stack([rng.permutation(E)[:k] for _ in range(M)]).astype(np.int32)).cuda(); w = torch.from_numpy(rng.random((M, k)).astype(np.float32)).cuda()
    mgr.forward(0, x[:40], ids[:40], w[:40])
    torch.empty((M, H), device="cuda")                               # (torch's own, for the result)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    mgr.forward(0, x, ids, w)
    torch.cuda.synchronize()
    need = (M * k + M) * (2 * I + 4 * H) + 431 * 2 * I * 4 + 215 * 2 * I * 4      # digits and results; gate and up of up to 431 rows on nine experts, and of the shared one's 215
    assert before - torch.cuda.mem_get_info()[0] <= need + (12 << 20)       # each buffer in whole pages of 2 MB
