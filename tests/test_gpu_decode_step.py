"""GPU parity of the fused decode step (encode new keys -> encode queries -> block top-k):
it must equal the separate operators, which are themselves checked against the CPU oracle,
and a HIP-graph replay of it must equal the eager result on every replay."""
import numpy as np
import pytest
import torch

from helpers import rng_for
from oracle import c_api

pytestmark = pytest.mark.gpu


def build(seed, B=4, Hq=32, Hkv=8, D=128, BS=128, nblk=6, per_head_w=True):
    from ucm_amd.sparse import HashEncoder

    rng = rng_for(seed)
    NB = B * nblk + 3
    W = torch.from_numpy(rng.standard_normal((Hkv, D, D) if per_head_w else (D, D))
                         .astype(np.float32)).to(torch.bfloat16).cuda()
    cache = torch.from_numpy(rng.integers(-2**31, 2**31 - 1, size=(NB, BS, Hkv, D // 32),
                                          dtype=np.int64).astype(np.int32)).cuda()
    table = torch.from_numpy(rng.permutation(NB)[: B * nblk].astype(np.int32).reshape(B, nblk)).cuda()
    lens = torch.from_numpy(rng.integers((nblk - 1) * BS + 1, nblk * BS + 1, size=B).astype(np.int32)).cuda()
    keys = torch.from_numpy(rng.standard_normal((B, Hkv, D)).astype(np.float32)).to(torch.bfloat16).cuda()
    qs = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(torch.bfloat16).cuda()
    # the new token of request b sits at position len-1
    pos = lens.to(torch.int64) - 1
    slots = table[torch.arange(B), (pos // BS)].to(torch.int64) * BS + pos % BS
    nw = Hkv if per_head_w else 1
    enc_k = HashEncoder(D, D, torch.bfloat16, torch.device("cuda:0"), num_weights=nw, heads_per_weight=1)
    enc_k.set_hash_weight(W)
    enc_q = HashEncoder(D, D, torch.bfloat16, torch.device("cuda:0"), num_weights=nw,
                        heads_per_weight=Hq // Hkv)
    enc_q.set_hash_weight(W)
    return W, cache, table, lens, keys, qs, slots, enc_k, enc_q


@pytest.mark.parametrize("per_head_w", [True, False])
def test_fused_step_equals_separate_operators_and_oracle(per_head_w):
    from ucm_amd.sparse import SparseDecodeStep, hamming_topk

    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(1, per_head_w=per_head_w)
    cache2 = cache.clone()
    B, Hq, Hkv, nblk, K = 4, 32, 8, 6, 3
    st = SparseDecodeStep(W, Hq, Hkv, B, nblk, K)
    idx, sc = st.step(keys, slots, qs, cache, table, lens)
    torch.cuda.synchronize()
    enc_k.compute_hash_and_cache(keys, slots, cache2, 128)
    qc = enc_q.compute_hash(qs, per_head=per_head_w).view(torch.int32)
    i2, s2 = hamming_topk(qc, cache2, table, lens, K)
    assert torch.equal(cache, cache2)
    assert torch.equal(st.q_codes, qc)
    assert torch.equal(idx, i2) and torch.equal(sc, s2)
    oi, osc = c_api.hamming_topk(qc.cpu().numpy().view(np.uint32), cache.cpu().numpy().view(np.uint32),
                                 table.cpu().numpy(), lens.cpu().numpy(), K)
    assert np.array_equal(idx.cpu().numpy(), oi) and np.array_equal(sc.cpu().numpy(), osc)


def test_bound_step_follows_tensor_contents():
    """bind() freezes the arguments, not the data: new queries in the same tensor give the new
    answer, identical to an unbound step()."""
    from ucm_amd.sparse import SparseDecodeStep

    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(3)
    B, Hq, Hkv, nblk, K = 4, 32, 8, 6, 3
    st = SparseDecodeStep(W, Hq, Hkv, B, nblk, K)
    run = st.bind(keys, slots, qs, cache, table, lens)
    i1, s1 = (t.clone() for t in run())
    e1, f1 = (t.clone() for t in st.step(keys, slots, qs, cache, table, lens))
    assert torch.equal(i1, e1) and torch.equal(s1, f1)
    qs.copy_(torch.flip(qs, dims=[0]))
    i2, s2 = (t.clone() for t in run())
    e2, f2 = (t.clone() for t in st.step(keys, slots, qs, cache, table, lens))
    assert torch.equal(i2, e2) and torch.equal(s2, f2)
    assert not torch.equal(s1, s2)


def test_step_without_new_keys_leaves_cache_untouched():
    from ucm_amd.sparse import SparseDecodeStep

    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(2)
    before = cache.clone()
    st = SparseDecodeStep(W, 32, 8, 4, 6, 2, reduce_heads=True, return_physical=True)
    idx, sc = st.step(None, None, qs, cache, table, lens)
    torch.cuda.synchronize()
    assert torch.equal(cache, before)
    qc = st.q_codes.cpu().numpy().view(np.uint32)
    oi, osc = c_api.hamming_topk(qc, cache.cpu().numpy().view(np.uint32), table.cpu().numpy(),
                                 lens.cpu().numpy(), 2, flags=c_api.F_REDUCE_HEADS | c_api.F_PHYSICAL)
    assert np.array_equal(idx.cpu().numpy(), oi) and np.array_equal(sc.cpu().numpy(), osc)


def test_graph_replays_match_eager_every_time():
    """Replay the captured step several times with eager work and synchronisations between
    the replays; inputs change between replays, so every replay must recompute."""
    from ucm_amd.sparse import SparseDecodeStep

    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(3)
    st = SparseDecodeStep(W, 32, 8, 4, 6, 3)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        st.step(keys, slots, qs, cache, table, lens)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st.step(keys, slots, qs, cache, table, lens)
    rng = rng_for(33)
    for rep in range(4):
        # new inputs written in place (the graph reads the same buffers)
        qs.copy_(torch.from_numpy(rng.standard_normal(tuple(qs.shape)).astype(np.float32)).to(torch.bfloat16))
        keys.copy_(torch.from_numpy(rng.standard_normal(tuple(keys.shape)).astype(np.float32)).to(torch.bfloat16))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        gi, gs, gc = st.out_idx.clone(), st.out_score.clone(), cache.clone()
        ei, es = st.step(keys, slots, qs, cache, table, lens)
        torch.cuda.synchronize()
        assert torch.equal(gi, ei) and torch.equal(gs, es) and torch.equal(gc, cache)
        _ = (qs.float() @ qs.float().transpose(1, 2)).sum().item()  # unrelated eager work


def test_argument_errors():
    from ucm_amd.sparse import SparseDecodeStep

    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(4)
    st = SparseDecodeStep(W, 32, 8, 4, 6, 3)
    with pytest.raises(ValueError):
        st.step(keys, slots, qs[:, :16], cache, table, lens)
    with pytest.raises(ValueError):
        st.step(keys, slots, qs.float(), cache, table, lens)
    with pytest.raises(ValueError):
        st.step(keys, slots, qs, cache, table.to(torch.int64), lens)
    with pytest.raises(ValueError):
        SparseDecodeStep(W[:3], 32, 8, 4, 6, 3)


@pytest.mark.parametrize("Hq,T", [(64, 4), (8, 4), (1, 0), (128, 4)])
def test_fused_latent_attention_step_equals_separate_operators_and_oracle(Hq, T):
    """MLA: nope (512) + rope (64) encoders, 18-word codes, one KV head; the fused call must
    leave the same codes in the cache and return the same blocks as the separate operators;
    the replayed HIP graph of it must agree with the eager call."""
    from ucm_amd.sparse import HashEncoder, SparseDecodeStepMLA, hamming_topk

    rng = rng_for(91 + Hq)
    B, BS, nblk, K = 4, 64, 20, 5
    NB = B * nblk + 3
    dev = torch.device("cuda:0")
    en = HashEncoder(512, 512, torch.bfloat16, dev)
    er = HashEncoder(64, 64, torch.bfloat16, dev)
    cache = torch.from_numpy(rng.integers(-2**31, 2**31 - 1, size=(NB, BS, 18), dtype=np.int64)
                             .astype(np.int32)).cuda()
    table = torch.from_numpy(rng.permutation(NB)[: B * nblk].astype(np.int32).reshape(B, nblk)).cuda()
    lens = torch.from_numpy(rng.integers((nblk - 1) * BS + 1, nblk * BS + 1, size=B).astype(np.int32)).cuda()
    bf = lambda shape: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(torch.bfloat16).cuda()
    kn, kr, qn, qr = bf((B, 512)), bf((B, 64)), bf((B, Hq, 512)), bf((B, Hq, 64))
    pos = lens.to(torch.int64) - 1
    slots = table[torch.arange(B), (pos // BS)].to(torch.int64) * BS + pos % BS
    cache2 = cache.clone()
    st = SparseDecodeStepMLA(en.hash_weights, er.hash_weights, Hq, B, nblk, K, block_size=BS,
                             sink_token=BS, recent_token=4 * BS, return_physical=True)
    args = (kn[:T] if T else None, kr[:T] if T else None, slots[:T] if T else None, qn, qr, cache, table, lens)
    idx, sc = st.step(*args)
    torch.cuda.synchronize()
    idx, sc = idx.clone(), sc.clone()
    # separate operators
    u8 = cache2.view(torch.uint8).unsqueeze(2)
    if T:
        en.compute_hash_and_cache(kn[:T, None], slots[:T], u8[..., :64], BS)
        er.compute_hash_and_cache(kr[:T, None], slots[:T], u8[..., 64:], BS)
    qc = torch.cat([en.compute_hash(qn), er.compute_hash(qr)], dim=-1).view(torch.int32)
    i2, s2 = hamming_topk(qc, cache2.unsqueeze(2), table, lens, K, BS, 4 * BS, return_physical=True)
    assert torch.equal(cache, cache2)
    assert torch.equal(st.q_codes, qc)
    assert torch.equal(idx, i2) and torch.equal(sc, s2)
    oi, osc = c_api.hamming_topk(qc.cpu().numpy().view(np.uint32),
                                 cache.cpu().numpy().view(np.uint32).reshape(NB, BS, 1, 18),
                                 table.cpu().numpy(), lens.cpu().numpy(), K, BS, 4 * BS, flags=c_api.F_PHYSICAL)
    assert np.array_equal(idx.cpu().numpy(), oi) and np.array_equal(sc.cpu().numpy(), osc)
    # graph replays (the step allocates nothing)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st.step(*args)
    for _ in range(3):
        st.out_idx.fill_(-7)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(st.out_idx, idx) and torch.equal(st.out_score, sc)


@pytest.mark.parametrize("B,Hq,R,T,dt", [
    (1, 1, 1, 1, torch.bfloat16), (1, 2, 2, 1, torch.float16),    # one row; the mean of two
    (2, 32, 2, 3, torch.bfloat16), (5, 16, 1, 5, torch.bfloat16),  # a whole row tile; two and a half
    (4, 128, 2, 33, torch.float16), (9, 64, 2, 40, torch.bfloat16),  # eight row tiles; nine, two tiles of keys
    (3, 48, 2, 2, torch.bfloat16), (2, 64, 4, 2, torch.bfloat16),  # 24 heads, means of four: the kernel of every form
])
@pytest.mark.parametrize("slots_i64", [False, True])
def test_latent_step_hashes_every_row(B, Hq, R, T, dt, slots_i64):
    """Codes of queries (means of R heads) and new keys against float64: a bit may differ only where the projection is
    within 1e-5 of its row's length of zero (sums of 512 products in fp32 are within 512 * 2^-24 = 3e-5 of the sum of
    their sizes, 0.8 / sqrt(512) of that bound for a random sign pattern).  Rows with gaps, a slot outside the cache."""
    from oracle import brute
    from ucm_amd.sparse.decode_step import GSADecodeStepMLA

    rng = rng_for(17 * B + Hq + R + T)
    BS, nblk = 64, 12
    NB = B * nblk + 2
    f = lambda *shape: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(dt).cuda()
    wn, wr, keys, qs = f(512, 512), f(64, 64), f(T, 640), f(B, Hq, 640)
    cache = torch.from_numpy(rng.integers(-2**31, 2**31 - 1, size=(NB, BS, 18), dtype=np.int64).astype(np.int32)).cuda()
    before = cache.cpu().numpy().view(np.uint32).reshape(NB * BS, 18)
    table = torch.from_numpy(rng.permutation(NB)[: B * nblk].astype(np.int32).reshape(B, nblk)).cuda()
    lens = torch.full((B,), nblk * BS, dtype=torch.int32, device="cuda")
    where = rng.permutation(NB * BS)[:T].astype(np.int64)
    if T > 1:
        where[T // 2] = -1 if slots_i64 else NB * BS
    slots = torch.from_numpy(where if slots_i64 else where.astype(np.int32)).cuda()
    st = GSADecodeStepMLA(wn, wr, Hq, R, B, nblk, 6 * BS, block_size=BS)
    st.step(keys[:, :512], keys[:, 512:576], slots, qs[..., :512], qs[..., 512:576], cache, table, lens)
    torch.cuda.synchronize()

    def agree(got, rows, first, w):
        x, W = rows.double().cpu().numpy(), w.double().cpu().numpy()
        diff = np.unpackbits((got[:, first:first + W.shape[1] // 32] ^ brute.hash_encode(x, W)).view(np.uint8), axis=-1, bitorder="little")
        assert not np.any(diff.astype(bool) & (brute.margins(x, W) >= 1e-5 * np.sqrt(x.shape[1])))

    means = qs.float().view(B, R, Hq // R, 640).mean(1).to(dt).view(-1, 640)
    codes = st.q_codes.cpu().numpy().view(np.uint32).reshape(-1, 18)
    agree(codes, means[:, :512], 0, wn)
    agree(codes, means[:, 512:576], 16, wr)
    after = cache.cpu().numpy().view(np.uint32).reshape(NB * BS, 18)
    ok = (where >= 0) & (where < NB * BS)
    agree(after[where[ok]], keys[torch.from_numpy(ok)][:, :512], 0, wn)
    agree(after[where[ok]], keys[torch.from_numpy(ok)][:, 512:576], 16, wr)
    rest = np.ones(NB * BS, bool)
    rest[where[ok]] = False
    assert np.array_equal(after[rest], before[rest])


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nn,Nr", [(512, 64), (64, 32), (128, 32), (256, 128), (512, 256), (1024, 512)])
def test_latent_step_of_any_width_and_rows_without_a_sign(R, dt, Nn, Nr):
    """Every number of column tiles of both parts, and rows of zeros, with a NaN and with an infinity among the keys and
    the queries (in their wide part, their narrow part or both): no bit set in the first two, and every code the one that
    the separate encoders give, which take the sums in the same order."""
    from ucm_amd.sparse import HashEncoder
    from ucm_amd.sparse.decode_step import GSADecodeStepMLA

    rng = rng_for(Nn + Nr + R)
    B, Hq, T, BS, nblk = 3, 32, 9, 64, 12
    NB, Wn = B * nblk, Nn // 32
    f = lambda *shape: torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(dt).cuda()
    wn, wr = f(512, Nn), f(64, Nr)
    parts = {512: (f(T, 512), f(B, R, Hq // R, 512)), 64: (f(T, 64), f(B, R, Hq // R, 64))}
    special = {512: (0, 1, 2), 64: (0, 3, 4)}  # rows of zeros, with a NaN, with an infinity
    for K, (k, q) in parts.items():
        zero, nan, inf = special[K]
        k[zero], q[1, :, zero] = 0, 0
        k[nan, K - 3] = q[0, R - 1, nan, 17] = float("nan")
        k[inf, 40] = q[2, R - 1, inf, K - 1] = float("inf")
    cache = torch.zeros((NB, BS, Wn + Nr // 32), dtype=torch.int32, device="cuda")
    table = torch.arange(NB, dtype=torch.int32, device="cuda").view(B, nblk)
    lens = torch.full((B,), nblk * BS, dtype=torch.int32, device="cuda")
    slots = torch.from_numpy(rng.permutation(NB * BS)[:T].astype(np.int64)).cuda()
    st = GSADecodeStepMLA(wn, wr, Hq, R, B, nblk, 6 * BS, block_size=BS)
    st.step(parts[512][0], parts[64][0], slots, parts[512][1].view(B, Hq, 512), parts[64][1].view(B, Hq, 64), cache, table, lens)
    torch.cuda.synchronize()
    codes = st.q_codes.view(B, Hq // R, -1)
    keys = cache.view(NB * BS, -1)[slots]
    for K, w, words in ((512, wn, slice(0, Wn)), (64, wr, slice(Wn, None))):
        k, q = parts[K]
        enc = HashEncoder(K, w.shape[1], dt, torch.device("cuda:0"))
        enc.set_hash_weight(w)
        zero, nan, _ = special[K]
        assert not keys[[zero, nan], words].any() and not codes[1, zero, words].any() and not codes[0, nan, words].any()
        assert torch.equal(keys[:, words], enc.compute_hash(k).view(torch.int32))
        means = (q.float().sum(1) / R).to(dt)
        assert torch.equal(codes[..., words], enc.compute_hash(means).view(torch.int32))


def select_long_rows(nblk, flips, BS, G, Wd=18):
    """Rows whose scores are G * (32 Wd - flips): every token of a block is the same, the query with as many bits turned."""
    from ucm_amd.sparse import hamming_topk

    rng = rng_for(nblk)
    B = 2
    q = np.broadcast_to(rng.integers(0, 2**32, (B, 1, Wd), dtype=np.uint32), (B, G, Wd)).copy()
    blocks = np.broadcast_to(q[:1, :1], (nblk, BS, Wd)).copy()
    for j in range(nblk):
        bits = np.zeros(32 * Wd, np.uint8)
        bits[rng.permutation(32 * Wd)[: flips[j]]] = 1
        blocks[j] ^= np.packbits(bits, bitorder="little").view(np.uint32)
    table = np.stack([rng.permutation(nblk), rng.permutation(nblk)]).astype(np.int32)
    lens = np.array([nblk * BS, (nblk - 3) * BS - 5], np.int32)
    t = lambda a: torch.from_numpy(a.view(np.int32)).cuda()
    for k in (1, 4, nblk // 3):
        gi, gs = hamming_topk(t(q), t(blocks).unsqueeze(2), t(table), t(lens), k, BS, 4 * BS, return_physical=True)
        oi, osc = c_api.hamming_topk(q, blocks[:, :, None], table, lens, k, BS, 4 * BS, flags=c_api.F_PHYSICAL)
        assert np.array_equal(gi.cpu().numpy(), oi) and np.array_equal(gs.cpu().numpy(), osc)


@pytest.mark.parametrize("nblk", [257, 512, 700, 2049])
@pytest.mark.parametrize("kind", ["ties", "spread", "outlier", "kept", "two", "64", "65"])
def test_selection_of_long_rows(nblk, kind):
    """Rows of every number of scores a thread, whose scores are all equal, anywhere in the range, close together but
    for one far below, blocks that equal the query beside those that are always kept (fewer and more than k), and few
    values: two, and on both sides of as many as have several bins each."""
    rng = rng_for(nblk + 1)
    flips = {"ties": np.full(nblk, 40), "spread": rng.integers(0, 577, nblk),
             "outlier": np.where(np.arange(nblk) == 77, 576, rng.integers(200, 205, nblk)),
             "kept": np.where(np.arange(nblk) % 5 == 2, 0, rng.integers(1, 300, nblk)),
             "two": 100 + np.arange(nblk) // 3 % 2, "64": 100 + np.arange(nblk) % 64, "65": 100 + np.arange(nblk) % 65}[kind]
    select_long_rows(nblk, flips, 64, 64 if kind in ("ties", "spread", "outlier", "kept") else 1)


@pytest.mark.parametrize("nblk", [300, 1100])
def test_selection_of_long_rows_in_three_steps(nblk):
    """240 heads of 1,536 bits: a range above 2^18, of which a step of 512 bins leaves 1,024 values and the next one two, so
    that the third counts in the first one's bins again."""
    flips = rng_for(nblk).integers(1, 1537, nblk)
    assert 240 * int(np.max(flips) - np.min(flips)) >= 2**18
    select_long_rows(nblk, flips, 16, 240, 48)


@pytest.mark.parametrize("G", [4, 8])
def test_separate_operators_under_graph_capture(G):
    """The operators a serving engine captures one by one (encode-and-cache, query hash, block
    top-k, per-token scores) in one HIP graph: every replay, with new inputs written in place and
    eager work between the replays, must equal the eager calls and the CPU checker.  G = 8 takes
    the bit-plane path (an extra kernel and its workspace inside the graph)."""
    from ucm_amd.sparse import hamming_score, hamming_topk

    Hkv, K = 8, 3
    W, cache, table, lens, keys, qs, slots, enc_k, enc_q = build(5, Hq=Hkv * G)
    from ucm_amd.sparse import HashEncoder

    enc_q = HashEncoder(128, 128, torch.bfloat16, torch.device("cuda:0"), num_weights=Hkv, heads_per_weight=G)
    enc_q.set_hash_weight(W)
    msl = table.shape[1] * 128

    def ops():
        enc_k.compute_hash_and_cache(keys, slots, cache, 128)
        qc = enc_q.compute_hash(qs, per_head=True).view(torch.int32)
        idx, sc = hamming_topk(qc, cache, table, lens, K)
        tok = hamming_score(cache, qc[:, None], table, lens, msl, 128, 256, False, out_int32=True)
        return qc, idx, sc, tok

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        g_out = ops()
    rng = rng_for(55 + G)
    for rep in range(3):
        qs.copy_(torch.from_numpy(rng.standard_normal(tuple(qs.shape)).astype(np.float32)).to(torch.bfloat16))
        keys.copy_(torch.from_numpy(rng.standard_normal(tuple(keys.shape)).astype(np.float32)).to(torch.bfloat16))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in g_out]
        gc = cache.clone()
        want = ops()
        torch.cuda.synchronize()
        assert torch.equal(gc, cache)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        oi, osc = c_api.hamming_topk(got[0].cpu().numpy().view(np.uint32), gc.cpu().numpy().view(np.uint32),
                                     table.cpu().numpy(), lens.cpu().numpy(), K)
        assert np.array_equal(got[1].cpu().numpy(), oi) and np.array_equal(got[2].cpu().numpy(), osc)
        ot = c_api.hamming_score(got[0].cpu().numpy().view(np.uint32), gc.cpu().numpy().view(np.uint32),
                                 table.cpu().numpy(), lens.cpu().numpy(), msl, 128, 256, False)
        assert np.array_equal(got[3].cpu().numpy(), ot)
        _ = (qs.float() @ qs.float().transpose(1, 2)).sum().item()  # unrelated eager work


@pytest.mark.parametrize("B,Hq,Hkv,D,BS,nblk,T,dtype,sink,recent", [
    (1, 8, 8, 128, 128, 40, 1, torch.bfloat16, None, None),   # no groups
    (3, 32, 8, 128, 128, 30, 3, torch.float16, None, None),
    (2, 64, 32, 128, 16, 61, 7, torch.bfloat16, 0, 16),       # no sink window, the most heads; more new keys than requests
    (5, 33, 1, 128, 48, 40, 9, torch.bfloat16, 48, 48),       # one head, an odd group, block size no power of two
    (2, 16, 2, 64, 1024, 12, 256, torch.bfloat16, 0, 1),      # the longest blocks, the most new keys
    (4, 20, 4, 64, 40, 50, 0, torch.float16, None, None),     # no new keys
    (16, 8, 4, 128, 64, 40, 16, torch.bfloat16, None, None),  # as many blocks as go this way
    (2, 10, 2, 64, 32, 300, 2, torch.bfloat16, 32, 64),       # a longer row for the selection
])
def test_small_step_scores_and_hashes_in_one_launch(B, Hq, Hkv, D, BS, nblk, T, dtype, sink, recent):
    """Steps of few blocks, whose scoring workgroups hash the queries: new keys inside scored blocks (their old
    codes must not count) and dropped ones, a block two requests share, unusable table entries, an empty request
    and lengths that end inside a block; the same codes, tables and lengths as the operators one by one."""
    from ucm_amd import _lib
    from ucm_amd.sparse import GSADecodeStep, HashEncoder

    rng = rng_for(B * 1009 + Hq * 31 + D + BS + T)
    NB, W = B * nblk + 2, D // 32
    w = torch.from_numpy(rng.standard_normal((D, D)).astype(np.float32)).to(dtype).cuda()
    cache = torch.from_numpy(rng.integers(0, 2**32, size=(NB, BS, Hkv, W), dtype=np.uint32).view(np.int32)).cuda()
    tab = rng.permutation(NB)[:B * nblk].astype(np.int32).reshape(B, nblk)
    lens = np.array([nblk * BS - (i * 37) % (nblk * BS // 2) for i in range(B)], np.int32)
    if B > 1:
        tab[1, 3] = tab[0, 2]
        lens[1] = nblk * BS - BS // 2
    if B > 2:
        lens[2] = 0
        tab[0, 4], tab[0, 5], tab[1, 0] = -1, NB, -3
    # new keys all over the first requests' blocks, each slot once
    slots = np.array([int(tab[0, 1 + i % (nblk - 2)]) * BS + (i * 7) % BS for i in range(T)], np.int64)
    slots = np.where((slots < 0) | (slots >= NB * BS), -1, slots)
    _, first = np.unique(slots, return_index=True)
    slots[np.setdiff1d(np.arange(T), first)] = -1
    if T:  # a code equal to its head's query code would be the best there is: old codes must not be seen
        q_at = slots[slots >= 0]
        cache.view(NB * BS, Hkv, W)[torch.from_numpy(q_at).cuda()] = 0
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(dtype).cuda()
    newk = torch.from_numpy(rng.standard_normal((T, Hkv, D)).astype(np.float32)).to(dtype).cuda() if T else None
    topk_tok = 8 * BS
    step = GSADecodeStep(w, Hq, Hkv, B, nblk, topk_tok, block_size=BS, sink_token=sink, recent_token=recent)
    expect_cache = cache.clone()
    enc = HashEncoder(D, D, dtype, torch.device("cuda:0"))
    enc.set_hash_weight(w)
    G = Hq // Hkv
    mean = q.view(B, Hkv, G, D)[:, :, 0].float()
    for g in range(1, G):  # the group's rows in order, as the step adds them
        mean = mean + q.view(B, Hkv, G, D)[:, :, g].float()
    mean = (mean * torch.tensor(1.0 / G, dtype=torch.float32)).to(dtype)
    qc = enc.compute_hash(mean).view(torch.int32)
    slot_t = torch.from_numpy(slots).cuda()
    if T:
        enc.compute_hash_and_cache(newk, slot_t, expect_cache, block_size=BS)
    new_table, new_lens = step.step(newk, slot_t if T else None, q, cache, torch.from_numpy(tab).cuda(), torch.from_numpy(lens).cuda())
    assert _lib.last_dispatch().startswith("encode_score<%d>+" % W)
    assert torch.equal(cache, expect_cache)
    assert torch.equal(step.q_codes.view(B, Hkv, W), qc.view(B, Hkv, W))
    oi, _ = c_api.hamming_topk(step.q_codes.cpu().numpy().view(np.uint32).reshape(B, Hkv, W),
                               cache.cpu().numpy().view(np.uint32), tab, lens, 8,
                               BS if sink is None else sink, 4 * BS if recent is None else recent,
                               flags=c_api.F_REDUCE_HEADS | c_api.F_PHYSICAL)
    expect = np.zeros((B, nblk), np.int32)
    for b in range(B):
        n = min(8, -(-int(lens[b]) // BS))
        expect[b, :n] = oi[b, 0, :n]
    assert np.array_equal(new_table.cpu().numpy(), expect)
    assert np.array_equal(new_lens.cpu().numpy(), c_api.update_seq_lens(lens, topk_tok, BS))


def _step_with_planted_keys(B, Hq, Hkv, D, BS, nblk, per):
    """A step whose list depends on the codes of its new keys: request b's new keys fill `per` slots each of two blocks
    outside the windows, all other codes of which are as far from the query as can be.  In one the slots hold the query's own
    code and the new keys are as far from it as can be (read too early, the block is the best there is), in the other
    the first of the new keys is the mean query itself.  The second request's table names a block of the first one."""
    from ucm_amd.sparse import HashEncoder

    dtype = torch.bfloat16
    rng = rng_for(B * 7919 + Hq * 31 + Hkv + D + BS + per)
    W, NB, G = D // 32, B * nblk, Hq // Hkv
    w = torch.from_numpy(rng.standard_normal((D, D)).astype(np.float32)).to(dtype).cuda()
    cache = torch.from_numpy(rng.integers(0, 2**32, size=(NB, BS, Hkv, W), dtype=np.uint32).view(np.int32)).cuda()
    tab = rng.permutation(NB).astype(np.int32).reshape(B, nblk)
    lens = np.full(B, nblk * BS, np.int32)
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(dtype).cuda()
    mean = q.view(B, Hkv, G, D)[:, :, 0].float()
    for g in range(1, G):
        mean = mean + q.view(B, Hkv, G, D)[:, :, g].float()
    mean = (mean * torch.tensor(1.0 / G, dtype=torch.float32)).to(dtype)
    enc = HashEncoder(D, D, dtype, torch.device("cuda:0"))
    enc.set_hash_weight(w)
    code = enc.compute_hash(mean).view(torch.int32).view(B, Hkv, W)
    keys, slots = [], []
    for b in range(B):
        stale, found = int(tab[b, 2 + b % 3]), int(tab[b, 6 + b % 2])
        cache[stale] = ~code[b]
        cache[found] = ~code[b]
        at = rng.choice(BS, size=(2, per), replace=False) if 2 * per <= BS else np.stack([rng.permutation(BS)[:per]] * 2)
        for i in range(per):
            cache[stale, int(at[0, i])] = code[b]
            keys += [-mean[b], mean[b] if i == 0 else -mean[b]]
            slots += [stale * BS + int(at[0, i]), found * BS + int(at[1, i])]
    if B > 1:
        tab[1, 4] = tab[0, 2]
    order = torch.from_numpy(rng.permutation(len(keys)))
    return w, enc, q, torch.stack(keys)[order.cuda()].contiguous(), torch.tensor(slots)[order].cuda(), cache, tab, lens


@pytest.mark.parametrize("B,Hq,Hkv,D,BS,nblk,per,one", [
    (1, 32, 8, 128, 128, 40, 1, True), (2, 8, 8, 128, 64, 40, 2, True), (1, 32, 8, 128, 32, 40, 14, True),  # up to 224 rows
    (3, 12, 1, 128, 128, 30, 32, True), (1, 32, 32, 128, 16, 40, 3, True),    # a head, as many as there may be
    (1, 32, 8, 64, 128, 40, 32, True), (2, 8, 2, 64, 1024, 14, 64, True),      # 64 bits: up to 512 rows
    (1, 32, 8, 128, 128, 40, 15, False), (1, 32, 8, 64, 128, 40, 33, False), (2, 64, 32, 128, 128, 40, 2, False),  # more
])
def test_new_keys_decide_which_blocks_are_listed(B, Hq, Hkv, D, BS, nblk, per, one):
    """Keys that the step writes itself count with their new codes, and the codes they replace not at all, in the kernel that
    hashes and scores at once and beyond the number of new keys up to which it is taken."""
    from ucm_amd import _lib
    from ucm_amd.sparse import GSADecodeStep

    w, enc, q, newk, slots, cache, tab, lens = _step_with_planted_keys(B, Hq, Hkv, D, BS, nblk, per)
    stale = cache.clone()
    expect_cache = cache.clone()
    enc.compute_hash_and_cache(newk, slots, expect_cache, block_size=BS)
    step = GSADecodeStep(w, Hq, Hkv, B, nblk, 6 * BS, block_size=BS, sink_token=BS, recent_token=2 * BS)
    table, _ = step.step(newk, slots, q, cache, torch.from_numpy(tab).cuda(), torch.from_numpy(lens).cuda())
    assert _lib.last_dispatch().startswith("encode_score<%d>+" % (D // 32)) == one
    assert torch.equal(cache, expect_cache)

    def listed(codes):
        oi, _ = c_api.hamming_topk(step.q_codes.cpu().numpy().view(np.uint32).reshape(B, Hkv, D // 32),
                                   codes.cpu().numpy().view(np.uint32), tab, lens, 6, BS, 2 * BS,
                                   flags=c_api.F_REDUCE_HEADS | c_api.F_PHYSICAL)
        return oi[:, 0]

    expect = listed(cache)
    assert np.array_equal(table.cpu().numpy()[:, :6], expect)
    # every request's list would be another one with the codes from before the step
    assert (listed(stale) != expect).any(axis=1).all()


@pytest.mark.parametrize("Hq,Hkv,D,BS,nblk,one", [
    (8, 8, 128, 128, 12, True), (4, 4, 128, 257, 12, True), (8, 8, 128, 383, 12, True), (2, 2, 128, 1024, 12, True),  # 1,024 codes and on
    (8, 8, 128, 1024, 9, True), (32, 32, 128, 1024, 9, True), (16, 16, 128, 512, 10, True),
    (16, 16, 128, 513, 10, False), (16, 16, 128, 1024, 9, False), (8, 8, 128, 1025, 9, False),
    (4, 2, 64, 511, 12, True), (16, 16, 64, 1024, 9, True), (32, 32, 64, 129, 12, True),
])
def test_codes_of_a_block_of_a_small_step(Hq, Hkv, D, BS, nblk, one):
    """Blocks of as many codes as a workgroup requests at first, a few more, and as many as there may be; lengths that end
    inside a block."""
    from ucm_amd import _lib
    from ucm_amd.sparse import GSADecodeStep

    rng = rng_for(Hq * 31 + Hkv + D + BS)
    B, W, dtype = 2, D // 32, torch.bfloat16
    w = torch.from_numpy(rng.standard_normal((D, D)).astype(np.float32)).to(dtype).cuda()
    cache = torch.from_numpy(rng.integers(0, 2**32, size=(B * nblk, BS, Hkv, W), dtype=np.uint32).view(np.int32)).cuda()
    tab = rng.permutation(B * nblk).astype(np.int32).reshape(B, nblk)
    lens = np.array([nblk * BS - 1, (nblk - 1) * BS - BS // 3], np.int32)
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(dtype).cuda()
    newk = torch.from_numpy(rng.standard_normal((B, Hkv, D)).astype(np.float32)).to(dtype).cuda()
    at = [2 * BS + BS - 1, 3 * BS]  # the last token of a block, the first of one
    slots = torch.tensor([int(tab[b, at[b] // BS]) * BS + at[b] % BS for b in range(B)])
    step = GSADecodeStep(w, Hq, Hkv, B, nblk, 5 * BS, block_size=BS, sink_token=0, recent_token=1)
    table, _ = step.step(newk, slots.cuda(), q, cache, torch.from_numpy(tab).cuda(), torch.from_numpy(lens).cuda())
    assert _lib.last_dispatch().startswith("encode_score<%d>+" % W) == one
    oi, _ = c_api.hamming_topk(step.q_codes.cpu().numpy().view(np.uint32).reshape(B, Hkv, W), cache.cpu().numpy().view(np.uint32),
                               tab, lens, 5, 0, 1, flags=c_api.F_REDUCE_HEADS | c_api.F_PHYSICAL)
    assert np.array_equal(table.cpu().numpy()[:, :5], oi[:, 0])


@pytest.mark.parametrize("D,Hq,B,nblk,one", [
    (128, 4, 4, 160, True), (128, 4, 4, 161, False), (64, 4, 4, 256, True), (64, 4, 4, 257, False), (64, 1, 9, 128, False),
    (64, 12, 9, 128, True), (64, 12, 5, 231, False),
])
def test_blocks_up_to_which_a_step_scores_and_hashes_at_once(D, Hq, B, nblk, one):
    """One generation of workgroups: 640 blocks of 128-bit codes, 1,024 of 64-bit ones on 256 compute units, 1,152 where the
    group's mean takes the encoder's launch longer."""
    from ucm_amd import _lib
    from ucm_amd.sparse import GSADecodeStep

    rng = rng_for(D + B + nblk)
    BS, W = 16, D // 32
    w = torch.from_numpy(rng.standard_normal((D, D)).astype(np.float32)).to(torch.bfloat16).cuda()
    cache = torch.from_numpy(rng.integers(0, 2**32, size=(B * nblk, BS, 1, W), dtype=np.uint32).view(np.int32)).cuda()
    tab = rng.permutation(B * nblk).astype(np.int32).reshape(B, nblk)
    lens = np.array([nblk * BS - 3 * b for b in range(B)], np.int32)
    q = torch.from_numpy(rng.standard_normal((B, Hq, D)).astype(np.float32)).to(torch.bfloat16).cuda()
    newk = torch.from_numpy(rng.standard_normal((B, 1, D)).astype(np.float32)).to(torch.bfloat16).cuda()
    slots = torch.tensor([int(tab[b, 7]) * BS + b for b in range(B)]).cuda()
    step = GSADecodeStep(w, Hq, 1, B, nblk, 12 * BS, block_size=BS)
    table, _ = step.step(newk, slots, q, cache, torch.from_numpy(tab).cuda(), torch.from_numpy(lens).cuda())
    assert _lib.last_dispatch().startswith("encode_score<%d>+" % W) == one
    oi, _ = c_api.hamming_topk(step.q_codes.cpu().numpy().view(np.uint32).reshape(B, 1, W), cache.cpu().numpy().view(np.uint32),
                               tab, lens, 12, BS, 4 * BS, flags=c_api.F_REDUCE_HEADS | c_api.F_PHYSICAL)
    assert np.array_equal(table.cpu().numpy()[:, :12], oi[:, 0])
