"""Strips of few rows per expert (krasis_amd/csrc/kr_prefill_strip.inc, kr_prefill_h.hip): the sort takes them where the experts' own rows are few, not where the average is, and the exact
ones give the bits of the decode kernels."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gemm_fast_gpu import _setup
from tests.test_gemm_ring_gpu import _prefill_mode
from tests.test_prefill_strips_cpu import plan
from tests.util import rand_bf16

pytestmark = pytest.mark.gpu
F = np.float32


def _cut(eng):
    from krasis_amd._lib import check
    n = (C.c_int(), C.c_int())
    check(eng._lib.kr_moe_prefill_tiles(eng._h, C.byref(n[0]), C.byref(n[1])))
    return n[0].value, n[1].value


def _forward(eng, torch, x, ids, w):
    from krasis_amd import _lib
    from krasis_amd._lib import check
    M, H = x.shape
    xt = torch.from_numpy(x.view(np.int16)).cuda(); it = torch.from_numpy(ids).cuda(); wt = torch.from_numpy(w).cuda()
    out = torch.empty((M, H), dtype=torch.float32, device="cuda")
    check(eng._lib.kr_moe_forward(eng._h, 0, xt.data_ptr(), it.data_ptr(), wt.data_ptr(), out.data_ptr(), M, ids.shape[1], _lib.KR_OUT_F32, 0, 1))
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _one_each(counts, k, rng):
    """ids [rows, k], one used slot a row: counts[e] rows of expert e in any order"""
    e = rng.permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.int32)
    ids = np.full((len(e), k), -1, np.int32)
    ids[np.arange(len(e)), rng.integers(0, k, len(e))] = e
    return ids


E = 64


@pytest.mark.parametrize("counts,exact,fast", [
    ([3] * E, "strips", "strips"),
    ([17] * 32 + [1] * 32, "strips", "tiles"),            # 96 strips of 16 for 64 tiles: as many as the exact rule takes
    ([17] * 33 + [1] * 31, "tiles", "tiles"),             # one more
    ([17] * 24 + [1] * 40, "strips", "strips"),           # 88 for 64: as many as the tolerance rule takes
    ([17] * 25 + [1] * 39, "strips", "tiles"),
    ([300, 299] + [0] * 62, "tiles", "tiles"),            # every row on the same two experts
    ([640] + [0] * 63, "tiles", "tiles"),
])
def test_the_cut_follows_the_experts_own_rows(counts, exact, fast):
    """at most ten rows an expert on average, where strips of 16 may be taken"""
    eng, experts, shared, rng, torch = _setup(256, 128, E, 1)
    ids = _one_each(counts, 1, rng)
    M = len(ids)
    assert M <= 10 * E
    x = rand_bf16(rng, (M, 256)); w = rng.random((M, 1)).astype(F)
    ref = _forward(eng, torch, x, ids, w)
    out = _prefill_mode(eng, torch, x, ids, w, 0)
    tiles, strips = _cut(eng)
    n = {"tiles": sum(-(-c // 64) for c in counts), "strips": sum(-(-c // 16) for c in counts)}
    assert (tiles, strips) == ((n["tiles"], 0) if exact == "tiles" else (0, n["strips"]))
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    tol = _prefill_mode(eng, torch, x, ids, w, 1)
    assert _cut(eng) == ((n["tiles"], 0) if fast == "tiles" else (0, n["strips"]))
    # rows and hidden values rounded to f16 once each, 2^-11 a value, in both products
    assert float(np.linalg.norm((tol - ref).astype(np.float64)) / np.linalg.norm(ref.astype(np.float64))) <= 2.0 ** -10


@pytest.mark.parametrize("per,strip", [(10, 16), (11, 32), (16, 32), (17, 64)])
@pytest.mark.parametrize("H,I", [(640, 384), (256, 128)])             # odd group counts in both products (the last step of a strip holds one); one step a strip
def test_exact_strips_are_the_decode_kernels_bits(H, I, per, strip):
    """rows an expert around the rules' lines (10: strips of 16, then of 32 to 16 with few experts), among them an expert without rows and ones of 1, 15 - 17 and 31 - 33"""
    eng, experts, shared, rng, torch = _setup(H, I, 20, 3)
    M = per * 20 // 3
    ids = np.argsort(rng.random((M, 20)), axis=1)[:, :3].astype(np.int32)
    ids[ids == 4] = -1
    ids[5, :] = -1
    x = rand_bf16(rng, (M, H)); w = rng.random((M, 3)).astype(F)
    out = _prefill_mode(eng, torch, x, ids, w, 0)
    tiles, strips = _cut(eng)
    counts = np.bincount(ids[ids >= 0], minlength=20)
    assert (strips == sum(-(-c // strip) for c in counts) and tiles == 0) if strip < 64 else (strips == 0 and tiles > 0), (tiles, strips, sorted(counts))
    assert np.array_equal(out.view(np.uint32), _forward(eng, torch, x, ids, w).view(np.uint32))


@pytest.mark.parametrize("counts", [(1, 15, 16, 17, 0, 2, 9, 8, 7, 3), (31, 32, 33, 1, 15, 16, 17, 0, 5, 10)])
def test_exact_strips_of_whole_and_ragged_tiles(counts):
    eng, experts, shared, rng, torch = _setup(384, 256, 10, 1)
    ids = _one_each(counts, 1, rng)
    x = rand_bf16(rng, (len(ids), 384)); w = rng.random((len(ids), 1)).astype(F)
    out = _prefill_mode(eng, torch, x, ids, w, 0)
    assert _cut(eng)[1] > 0
    assert np.array_equal(out.view(np.uint32), _forward(eng, torch, x, ids, w).view(np.uint32))


# (strips a wave of the whole rounds, of the rest, tiles in whole rounds; none where all are alike) of the two products
@pytest.mark.parametrize("E,per,strip,cuts", [(250, 12, 32, (None, None)), (257, 12, 32, ((4, 1, 256), (2, 1, 256))), (300, 12, 32, ((4, 1, 256), (2, 1, 256))),
                                              (520, 6, 16, ((4, 1, 512), (2, 1, 512))), (576, 6, 16, ((4, 1, 512), (2, 1, 512))), (640, 6, 16, (None, (2, 1, 512)))])
def test_exact_strips_whose_last_round_is_cut(E, per, strip, cuts):
    """tiles around what the chip holds (256 workgroups of 32 rows, 512 of 16): whole rounds with several strips a wave, and the tiles that are left, among them none, in smaller pieces"""
    import torch
    from krasis_amd import KrasisEngine, ModelConfig
    from tests.util import make_experts, upload
    rng = np.random.default_rng(E)
    few = make_experts(rng, 7, 512, 512, 4)
    eng = KrasisEngine(); eng.configure(ModelConfig(512, 512, E, 1, 1, 0, 1.0))
    upload(eng, 0, [few[e % 7] for e in range(E)], None)
    counts = np.full(E, per); counts[3], counts[8] = 0, strip + 1
    ids = _one_each(counts, 1, rng)
    x = rand_bf16(rng, (len(ids), 512)); w = rng.random((len(ids), 1)).astype(F)
    out = _prefill_mode(eng, torch, x, ids, w, 0)
    assert _cut(eng) == (0, E)                               # one tile an expert, one expert without, one with two
    most = len(ids) // strip + E + 1
    for N, want in ((1024, cuts[0]), (512, cuts[1])):
        (first, others, whole), places = plan(strip, N, 512, most, E)
        assert ((first, others, whole) == want) if want else (first == others or whole == E), (N, first, others, whole)
    assert np.array_equal(out.view(np.uint32), _forward(eng, torch, x, ids, w).view(np.uint32))


@pytest.mark.parametrize("Ms,ret_bf16", [([20, 12], False), ([20, 12], True), ([3, 0], False)])
def test_scattered_rows_of_expert_parallel_ranks(Ms, ret_bf16):
    """nine rows a local expert, each row stored at the place that it came from, in f32 and in bf16"""
    import tests.test_ep_gpu as ep
    ep.test_library_expert_parallel_loopback_equals_single_engine(2, Ms, ret_bf16, False)


@pytest.mark.parametrize("M", [2, 16, 17])
def test_up_to_sixteen_tokens(M):
    """strips whatever the rows, also where tokens name an expert twice and it has a second strip; one token more, and the experts' own rows decide"""
    eng, experts, shared, rng, torch = _setup(256, 128, 20, 3)
    x = rand_bf16(rng, (M, 256)); w = rng.random((M, 3)).astype(F)
    ids = np.full((M, 3), 7, np.int32); ids[:, 2] = 9; ids[0, 1] = -1
    out = _prefill_mode(eng, torch, x, ids, w, 0)
    rows = (2 * M - 1, M)
    assert _cut(eng) == ((0, sum(-(-r // 16) for r in rows)) if M <= 16 else (2, 0))
    ref = _forward(eng, torch, x, ids, w)
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32))
    tol = _prefill_mode(eng, torch, x, ids, w, 1)
    assert (_cut(eng)[1] > 0) == (M <= 16)
    assert float(np.linalg.norm((tol - ref).astype(np.float64)) / np.linalg.norm(ref.astype(np.float64))) <= 2.0 ** -10
