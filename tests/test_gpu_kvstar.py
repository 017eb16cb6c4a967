"""GPU parity: KVStar block retrieval (ucm_kvstar_topk through the kvstar_retrieve mirror)
against the CPU checker.

Tolerance: block scores are sums of fp32 softmax probabilities; the GPU adds the q.k partial
products and the exponentials in a different order than the checker's sequential loops, and its
expf differs from libm's by a few ulp.  Scores must agree within 2e-5 relative + 1e-7 absolute,
and where the returned block numbers differ the two blocks' checker scores must differ by less
than that tolerance (a tie within rounding).
"""
import numpy as np
import pytest
import torch

from oracle import brute, c_api
from ucm_amd.sparse import kvstar_retrieve

pytestmark = pytest.mark.gpu

RTOL, ATOL = 2e-5, 1e-7


def make(seed, X, Hq, Hkv, d, n, M, scale=0.5, d_orig=None):
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal((X, Hq, d_orig or d)) * scale).astype(np.float16)
    k = (rng.standard_normal((n, M, Hkv, d)) * scale).astype(np.float16)
    return q, k


def run_gpu(q, k, pr, topk):
    dev = torch.device("cuda:0")
    idx, sc = kvstar_retrieve.kvstar_topk(
        torch.from_numpy(q).to(dev), torch.from_numpy(k).to(dev),
        torch.from_numpy(pr).to(dev) if pr is not None else None, topk)
    torch.cuda.synchronize()
    return idx.cpu().numpy().astype(np.int64), sc.cpu().numpy()


def check(q, k, pr, topk):
    gi, gs = run_gpu(q, k, pr, topk)
    oi, osc, allsc = c_api.kvstar_topk(q, k, topk, pr)
    assert gi.shape == oi.shape
    tol = ATOL + RTOL * np.abs(osc)
    assert np.all(np.abs(gs - osc) <= tol), (gs, osc)
    assert np.all(np.diff(gs) <= 0)
    assert len(set(gi.tolist())) == gi.size
    for t in np.nonzero(gi != oi)[0]:
        assert abs(allsc[gi[t]] - allsc[oi[t]]) <= 2 * tol[t]
    # the returned score is the score of the returned block
    assert np.all(np.abs(gs - allsc[gi]) <= ATOL + RTOL * np.abs(allsc[gi]))


@pytest.mark.parametrize("X,Hq,Hkv,d,n,M,topk", [
    (1, 4, 4, 16, 7, 1, 3),        # MHA, one representative per block
    (3, 8, 2, 32, 24, 4, 5),       # GQA 4:1
    (8, 32, 8, 128, 100, 2, 16),   # Llama-like heads
    (5, 6, 3, 20, 40, 3, 8),       # head dim not a multiple of 8: scalar K loads
    (2, 4, 1, 64, 300, 1, 300),    # MQA, every block returned
    (17, 8, 8, 128, 513, 2, 64),   # more than one row tile, blocks past one workgroup
    (1, 1, 1, 8, 1, 1, 1),         # smallest problem
    (20, 8, 2, 32, 70, 3, 9),      # 80 query rows per KV head: three row tiles, ragged last tiles
    (3, 4, 2, 48, 33, 1, 5),       # three k-steps, one representative past a 32-wide tile
])
def test_matches_checker(X, Hq, Hkv, d, n, M, topk):
    q, k = make(X * 1000 + n, X, Hq, Hkv, d, n, M)
    check(q, k, None, topk)


@pytest.mark.parametrize("X,Hq,Hkv,d,n,M,topk", [
    (8, 8, 2, 32, 40, 31, 7),      # 32 query rows per KV head: whole tiles; one short of a tile of representatives
    (9, 8, 2, 64, 40, 32, 7),      # a row more than a tile; a block is a tile of representatives
    (3, 6, 2, 128, 9, 33, 9),      # a block of two tiles, the second with one representative
    (2, 4, 2, 32, 300, 3, 20),     # ten blocks share a tile
    (1, 2, 1, 64, 1, 100, 1),      # one block of several tiles
    (2, 4, 4, 32, 33, 63, 33),     # an odd number of row tiles per workgroup pair, chunks that end inside a tile
    (40, 64, 2, 32, 12, 2, 12),    # 2560 rows: statistics in two batches
    (2, 4, 2, 24, 21, 16, 5),      # head dim of one and a half k-steps
    (2, 4, 2, 256, 21, 16, 5),     # head dim above what is kept packed
    (1, 2, 2, 32, 70, 256, 11),    # more tiles than two per wave and chunk
])
def test_edges_of_the_tiles(X, Hq, Hkv, d, n, M, topk):
    q, k = make(X * 100 + n + d, X, Hq, Hkv, d, n, M)
    check(q, k, None, topk)


def test_far_scores_keep_their_order():
    """Blocks whose every probability lies far below the largest (e^-60 to e^-95) keep the order of
    their masses, down into the denormal range.  Relative tolerance: the scores' own rounding, 2^-24 of
    their size (95), moves a probability by 95 * 2^-24 < 6e-6; below 1e-38 one step of a denormal."""
    n, d = 36, 32
    q = np.zeros((1, 1, d), np.float16)
    q[0, 0, 0] = 8.0
    k = np.zeros((n, 1, 1, d), np.float16)
    k[:, 0, 0, 0] = -np.arange(n) * 2.65 / 8.0
    gi, gs = run_gpu(q, k, None, n)
    s = (q.astype(np.float64)[0, 0] @ k.astype(np.float64)[:, 0, 0].T)
    ref = np.exp(s - s.max()) / np.exp(s - s.max()).sum()
    assert gi.tolist() == list(range(n))
    assert np.all(np.abs(gs - ref) <= 1e-5 * ref + 2e-45)


@pytest.mark.parametrize("base", [-1.8e8, -1.92e8, -3.2e8, -4.0e9, 1.4e9, 1.6e9, 4.0e9])
@pytest.mark.parametrize("d,M", [(32, 1), (32, 3), (64, 40), (24, 3)])
def test_scores_of_any_finite_size(base, d, M):
    """Rows whose scores all lie near `base` (finite fp16 inputs reach 4.3e9 in one channel), beside a row of
    ordinary ones.  One channel makes the base, one adds steps of one fp32 unit of it: every product and sum
    is exact in any order, so the rows compare with the checker's at the usual tolerance."""
    n, rng = 45, np.random.default_rng(int(abs(base)) % 1000 + d)
    ulp = float(np.spacing(np.float32(abs(base))))
    a = 64.0 * round(abs(base) / 64 / 61440)         # times 61440 = 2^12 * 15: a multiple of 2^18
    q = np.zeros((2, 2, d), np.float16)
    q[:, :, 0], q[:, :, 1] = np.copysign(a, base), ulp
    q[1, 1, 0], q[1, 1, 1] = 0.0, 0.25               # an ordinary row
    k = np.zeros((n, M, 1, d), np.float16)
    k[..., 0] = 61440.0
    k[..., 1] = rng.integers(0, 4, (n, M, 1))
    assert a * 61440.0 + 3 * ulp != a * 61440.0 and abs(a * 61440 / abs(base) - 1) < 0.01
    check(q, k, None, n)


@pytest.mark.parametrize("n,M,d", [(40, 1, 32), (33, 3, 32), (30, 64, 64), (70, 20, 128), (40, 3, 24), (33, 33, 96)])
@pytest.mark.parametrize("what", ["nan", "+inf", "-inf", "nan_lane", "all_-inf"])
def test_infinite_and_undefined_scores(what, n, M, d):
    """As the checker has it: exponentials of the distance to the row's largest score, which passes over NaN
    (the checker's also does unless its first score is one); a row whose sum is NaN is not normalised; a row
    of minus infinities has NaN everywhere.  Blocks with a NaN score come last, in block order."""
    q, k = make(n + M + d, 2, 4, 2, d, n, M)
    q = np.abs(q) + np.float16(0.125)                # no zero times infinity
    flat = k.reshape(n * M, 2, d)
    S = n * M
    for s in (S // 3, S - 1):
        if what == "nan":
            flat[s, 0, 3] = np.nan                   # KV head 0 only: the other head's rows stay normalised
        elif what == "nan_lane":
            t = max(32, s - s % 32)                  # a tile of representatives, not the first: all scores of a lane
            flat[t:t + 32, 0, 3] = np.nan
        elif what == "+inf":
            flat[s, 0, 3] = np.inf
        elif what == "-inf":
            flat[s, 0, 3] = -np.inf
        else:
            flat[:, 0, 3] = -np.inf
    gi, gs = run_gpu(q, k, None, n)
    _, _, ref = c_api.kvstar_topk(q, k, n)
    undefined = np.isnan(ref)
    assert undefined.any() == (what != "-inf") and (undefined.all() == (what == "all_-inf"))
    got = np.zeros(n, np.float32)
    got[gi] = gs
    assert sorted(gi.tolist()) == list(range(n)) and np.array_equal(np.isnan(got), undefined)
    ok = ~undefined
    assert np.all(np.abs(got[ok] - ref[ok]) <= ATOL + RTOL * np.abs(ref[ok]))
    tail = gi[int(ok.sum()):]
    assert tail.tolist() == np.flatnonzero(undefined).tolist()


@pytest.mark.parametrize("d", [8, 17, 31, 32, 33, 48, 64, 80, 95, 96, 100, 112, 128, 130, 256, 512, 513, 1024])
@pytest.mark.parametrize("M", [3, 40])
def test_head_dimensions(d, M):
    """Every remainder of the k-steps (groups of four, two, one and a partial one), a query row of more
    channels than the keys have, and rows that start at odd multiples of two bytes."""
    Hkv, d_orig = 2, d + 5
    rng = np.random.default_rng(d)
    q, k = make(d * 10 + M, 3, 6, Hkv, d, 41, M, scale=0.5 if d < 200 else 0.25 if d < 500 else 0.15, d_orig=d_orig)
    pr = np.stack([np.sort(rng.permutation(d_orig)[:d]) for _ in range(Hkv)]).astype(np.int64)
    check(q, k, pr, 13)
    check(np.ascontiguousarray(q[..., :d]), k, None, 13)


@pytest.mark.parametrize("d", [32, 64, 100, 128, 256])
def test_probabilities_add_up_at_large_scores(d):
    """Scores of several 10,000 are steps of 2^-9 apart: the kernels that sum a row's exponentials and the
    block's probabilities take the same q.k, or rows would add up to e^(2^-9) and not to 1."""
    q, k = make(d, 4, 8, 2, d, 30, 40, scale=60.0)
    _, gs = run_gpu(q, k, None, 30)
    assert abs(gs.astype(np.float64).sum() - 32) < 32 * 1e-5


def test_sharp_softmax():
    # larger logits: a few representatives take most of the mass
    q, k = make(11, 4, 8, 4, 64, 200, 2, scale=1.5)
    check(q, k, None, 10)


def test_channel_pruning():
    rng = np.random.default_rng(12)
    Hkv, d_orig, d = 2, 128, 96
    q, k = make(12, 4, 8, Hkv, d, 64, 2, d_orig=d_orig)
    pr = np.stack([np.sort(rng.permutation(d_orig)[:d]) for _ in range(Hkv)]).astype(np.int64)
    check(q, k, pr, 12)


def test_against_float64_formulation_at_llama_shape():
    # a size the sequential checker would take long on: 8 query tokens x 32 heads against 4096
    # blocks x 2 representatives, compared with the float64 library formulation
    q, k = make(13, 8, 32, 8, 128, 4096, 2, scale=0.3)
    gi, gs = run_gpu(q, k, None, 64)
    ref = brute.kvstar_block_scores(q, k)
    assert np.allclose(gs, ref[gi], rtol=RTOL, atol=ATOL)
    kth = np.sort(ref)[::-1][63]
    assert np.all(ref[gi] >= kth - (ATOL + RTOL * kth))
    assert gs.sum() <= 8 * 32 * (1 + 1e-5)


@pytest.mark.parametrize("X,Hq,Hkv,d,n,M", [
    (1, 1, 1, 64, 1, 16), (2, 8, 8, 32, 3, 16),       # half a tile of representatives; one and a half
    (1, 6, 3, 128, 5, 16), (3, 6, 3, 64, 33, 32),     # an odd number of row tiles; of tiles of representatives
    (9, 32, 8, 32, 256, 16), (2, 4, 4, 32, 257, 32),   # a row's blocks in eight loads of the merging threads, one more
    (1, 8, 8, 32, 512, 16), (1, 8, 8, 32, 513, 16),
    (1, 8, 8, 32, 1024, 16), (1, 8, 8, 32, 1025, 16),  # the most blocks of 16 taken once, and one more
    (1, 2, 1, 32, 1025, 32), (1, 2, 1, 32, 2048, 64), (1, 2, 1, 32, 2049, 64),  # loaded twice; the most that are ranked
    (17, 8, 4, 128, 40, 64), (2, 4, 2, 64, 21, 128), (2, 4, 2, 32, 65, 256), (2, 4, 2, 32, 9, 320),
])
def test_blocks_whose_scores_are_taken_once(X, Hq, Hkv, d, n, M):
    """Against float64: 16, 32, 64, 128 and 256 representatives on both sides of where such blocks leave the
    general path.  Half of the blocks lie e^-60 below the others."""
    q, k = make(X + n + M + d, X, Hq, Hkv, d, n, M)
    q[..., 0] = 8.0
    k[..., 0] = np.where(np.arange(n) % 2 == 1, -7.5, 0.0)[:, None, None]
    gi, gs = run_gpu(q, k, None, n)
    ref = brute.kvstar_block_scores(q, k)
    assert sorted(gi.tolist()) == list(range(n)) and np.all(np.diff(gs) <= 0)
    assert np.all(np.abs(gs - ref[gi]) <= RTOL * ref[gi] + 2e-45)


@pytest.mark.parametrize("X,Hq,Hkv,d,d_orig,n,M", [
    (8, 32, 8, 32, 128, 253, 64),                      # 32k tokens, a quarter of the channels
    (5, 28, 4, 64, 100, 40, 32), (8, 28, 4, 32, 45, 70, 16), (3, 6, 2, 128, 130, 21, 192),  # seven and three heads to a group
    (2, 14, 2, 32, 64, 33, 192), (9, 20, 4, 64, 64, 25, 16), (1, 12, 1, 128, 160, 17, 256), (8, 8, 8, 32, 33, 9, 128),
])
def test_pruned_channels_and_any_group_taken_once(X, Hq, Hkv, d, d_orig, n, M):
    """Against float64: channels in any order, some twice, and some outside the query row, which count as its ends."""
    rng = np.random.default_rng(n + d)
    q, k = make(X * 7 + n, X, Hq, Hkv, d, n, M, scale=0.5 if d < 128 else 0.3, d_orig=d_orig)
    pr = rng.integers(0, d_orig, (Hkv, d))
    pr[:, 3], pr[-1, d // 2], pr[0, d - 1] = -2, d_orig, d_orig + 1000
    gi, gs = run_gpu(q, k, pr, n)
    ref = brute.kvstar_block_scores(q, k, np.clip(pr, 0, d_orig - 1))
    assert sorted(gi.tolist()) == list(range(n)) and np.all(np.diff(gs) <= 0)
    assert np.all(np.abs(gs - ref[gi]) <= RTOL * ref[gi])


@pytest.mark.parametrize("Hq,n", [(32767, 4), (32768, 8), (40000, 4), (65535, 3)])
def test_as_many_heads_to_a_group_as_are_taken(Hq, n):
    """Group sizes on both sides of 2^15 and the largest, against float64: blocks of very different mass."""
    q, k = make(Hq, 1, Hq, 1, 32, n, 16)
    k *= np.arange(1, n + 1, dtype=np.float16)[:, None, None, None] * np.float16(0.5)
    gi, gs = run_gpu(q, k, None, n)
    ref = brute.kvstar_block_scores(q, k)
    assert np.ptp(ref) > 0.1 * ref.mean()
    assert gi.tolist() == np.argsort(-ref, kind="stable").tolist()
    assert np.all(np.abs(gs - ref[gi]) <= RTOL * ref[gi])


@pytest.mark.parametrize("M", [16, 32, 128])
@pytest.mark.parametrize("what", ["nan", "+inf", "-inf", "nan_lane", "all_-inf"])
def test_infinite_and_undefined_scores_taken_once(what, M):
    test_infinite_and_undefined_scores(what, 300, M, 64 if M == 16 else 32)  # (two row tiles of 16 x 32 take the general path)


@pytest.mark.parametrize("base", [-3.2e8, 4.0e9])
@pytest.mark.parametrize("d,M", [(64, 16), (128, 16), (32, 32), (64, 32), (128, 64)])
def test_scores_of_any_finite_size_taken_once(base, d, M):
    test_scores_of_any_finite_size(base, d, M)


@pytest.mark.parametrize("asked,called", [
    ((8, 32, 2049, 64), (8, 32, 8, 32, 2048, 64)),   # one block less, and the blocks' products are taken once
    ((8, 32, 2049, 64), (8, 32, 8, 32, 300, 64)), ((8, 32, 513, 48), (8, 32, 8, 32, 513, 32)),
    ((16, 64, 2000, 64), (1, 64, 8, 32, 2000, 64)),  # fewer query tokens
    ((8, 32, 2000, 64), (8, 32, 8, 32, 2000, 64)), ((2, 4, 257, 32), (2, 4, 1, 512, 256, 32)),
    ((2, 4, 129, 64), (2, 4, 2, 256, 128, 64)),      # 65 chunks of four tiles would be asked for, in fives they are 52
])
def test_a_buffer_asked_for_at_a_larger_shape(asked, called):
    """The C call takes it, answers rightly and writes nothing behind it."""
    from ucm_amd import _lib

    X, Hq, Hkv, d, n, M = called
    size = _lib.lib().ucm_kvstar_topk_workspace_bytes(*asked)
    q, k = make(n, X, Hq, Hkv, d, n, M, scale=0.5 if d < 200 else 0.2)
    tq, tk = torch.from_numpy(q).cuda(), torch.from_numpy(k).cuda()
    ws = torch.full((size + 4096,), 0x5a, dtype=torch.uint8, device="cuda")
    idx, sc = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, dtype=torch.float32, device="cuda")
    rc = _lib.lib().ucm_kvstar_topk(tq.data_ptr(), X, Hq, d, tk.data_ptr(), n, M, Hkv, d, None, n, idx.data_ptr(), sc.data_ptr(),
                                    ws.data_ptr(), size, _lib.stream_ptr(tq.device))
    _lib.check(rc)
    ref = brute.kvstar_block_scores(q, k)
    gi, gs = idx.cpu().numpy(), sc.cpu().numpy()
    assert sorted(gi.tolist()) == list(range(n)) and np.all(np.abs(gs - ref[gi]) <= ATOL + RTOL * ref[gi])
    assert bool((ws[size:] == 0x5a).all())


def test_long_rows_in_two_batches_of_statistics():
    # 2560 query rows; against float64, as the checker adds a block's 102,400 probabilities one by one
    q, k = make(40, 40, 64, 2, 130, 9, 40, scale=0.5)
    gi, gs = run_gpu(q, k, None, 9)
    ref = brute.kvstar_block_scores(q, k)
    assert np.allclose(gs, ref[gi], rtol=RTOL, atol=ATOL) and np.all(np.diff(gs) <= 0)


def test_equal_scores_come_out_in_ascending_block_order():
    q, _ = make(14, 2, 4, 2, 16, 1, 1)
    k = np.full((8, 2, 2, 16), 0.25, np.float16)
    gi, gs = run_gpu(q, k, None, 3)
    assert gi.tolist() == [0, 1, 2]
    assert np.allclose(gs, 2 * 4 / 8, rtol=1e-6)


def test_module_api_like_the_reference_call_site():
    q, k = make(15, 3, 8, 2, 32, 50, 2)
    kvstar_retrieve.Setup(kvstar_retrieve.SetupParam(cpuNumaIds=[0], bindInfo=[(0, 0)],
                                                     deviceType=kvstar_retrieve.CPU,
                                                     totalTpSize=1, localRankId=0))
    tid = kvstar_retrieve.AsyncRetrieveByCPU(torch.from_numpy(q), torch.from_numpy(k), None, 6, 42,
                                             kvstar_retrieve.CPU)
    assert kvstar_retrieve.Wait(tid) == 0
    res = kvstar_retrieve.GetTaskResult(tid)
    assert res["status"] == "SUCCESS"
    oi, _, _ = c_api.kvstar_topk(q, k, 6)
    assert res["data"] == oi.tolist()
    assert kvstar_retrieve.Wait(tid) != 0          # the waiter is gone after the first Wait
    assert kvstar_retrieve.GetTaskResult(10 ** 9) is None
    # topK above the number of blocks returns every block
    tid = kvstar_retrieve.AsyncRetrieveByCPU(torch.from_numpy(q), torch.from_numpy(k), None, 80, 42,
                                             kvstar_retrieve.CPU)
    kvstar_retrieve.Wait(tid)
    assert sorted(kvstar_retrieve.GetTaskResult(tid)["data"]) == list(range(50))


def test_failures_are_reported_on_the_task():
    q, k = make(16, 2, 6, 4, 16, 10, 1)  # 6 q heads over 4 kv heads
    tid = kvstar_retrieve.AsyncRetrieveByCPU(torch.from_numpy(q), torch.from_numpy(k), None, 3, 1,
                                             kvstar_retrieve.CPU)
    assert kvstar_retrieve.Wait(tid) != 0
    res = kvstar_retrieve.GetTaskResult(tid)
    assert res["status"] == "FAILURE" and "divisible" in res["error"]
    q, k = make(17, 2, 4, 2, 16, 10, 1, d_orig=32)  # head dims differ and no pruning index
    tid = kvstar_retrieve.AsyncRetrieveByCPU(torch.from_numpy(q), torch.from_numpy(k), None, 3, 1,
                                             kvstar_retrieve.CPU)
    kvstar_retrieve.Wait(tid)
    assert "Dimension mismatch" in kvstar_retrieve.GetTaskResult(tid)["error"]
