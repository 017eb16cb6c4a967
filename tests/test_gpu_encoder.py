"""GPU parity: the HIP sign-hash encoder against the CPU oracle.

Tolerance rule (the only floating-point tolerance in the suite): a hash bit may differ from
the oracle only where |projection| < 1e-2 * ||x||; everywhere else it must be identical.
The oracle used for the comparison accumulates in float64.
"""
import numpy as np
import pytest
import torch

from helpers import rng_for
from oracle import brute, c_api

pytestmark = pytest.mark.gpu

MARGIN_TOL = 1e-2


def bf16_round(a):
    return torch.from_numpy(np.asarray(a, np.float32)).to(torch.bfloat16)


def assert_codes_match(codes_u8, x32, W32):
    """codes_u8 [M, N/8] from the GPU; x32 [M,K], W32 [K,N] the exact values the GPU saw."""
    ref = brute.hash_encode(x32, W32).view(np.uint8)
    got = np.ascontiguousarray(codes_u8)
    if np.array_equal(got, ref):
        return 0
    diff_bits = np.unpackbits(got ^ ref, axis=-1, bitorder="little").astype(bool)
    marg = brute.margins(x32, W32)
    assert not np.any(diff_bits & (marg >= MARGIN_TOL)), "bit flipped outside the margin"
    return int(diff_bits.sum())


def make_encoder(K, N, dtype, W, n_w=1, hpw=1):
    from ucm_amd.sparse import HashEncoder

    enc = HashEncoder(K, N, dtype, torch.device("cuda:0"), num_weights=n_w, heads_per_weight=hpw)
    enc.set_hash_weight(W.to(dtype).cuda())
    return enc


def test_bit_and_byte_order_with_identity_weights():
    K = N = 128
    enc = make_encoder(K, N, torch.bfloat16, torch.eye(K))
    x = torch.zeros(5, K)
    x[0, 0] = 1.0
    x[1, 9] = 2.0
    x[2, 37] = 0.5
    x[2, 3] = -1.0
    x[3, 127] = 3.0
    x[4, :] = -1.0
    codes = enc.compute_hash(x.to(torch.bfloat16).cuda()).cpu().numpy()
    words = np.ascontiguousarray(codes).view("<u4")
    assert words[0].tolist() == [1, 0, 0, 0]
    assert words[1].tolist() == [1 << 9, 0, 0, 0]
    assert words[2].tolist() == [0, 1 << 5, 0, 0]
    assert words[3].tolist() == [0, 0, 0, 1 << 31]
    assert words[4].tolist() == [0, 0, 0, 0]
    assert codes[1, 1] == 2  # byte 1, bit 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(1, 128, 128), (33, 128, 128), (300, 128, 128),
                                   (70, 64, 64), (40, 256, 128), (50, 512, 256), (17, 128, 96)])
def test_compute_hash_matches_oracle(dtype, M, K, N):
    rng = rng_for(1000 + M + K + N)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dtype)
    W = torch.from_numpy(rng.standard_normal((K, N)).astype(np.float32)).to(dtype)
    enc = make_encoder(K, N, dtype, W)
    codes = enc.compute_hash(x.cuda())
    assert codes.dtype == torch.uint8 and tuple(codes.shape) == (M, N // 8)
    assert_codes_match(codes.cpu().numpy(), x.float().numpy(), W.float().numpy())


def test_leading_dims_and_negation():
    rng = rng_for(7)
    x = bf16_round(rng.standard_normal((3, 5, 128)))
    W = bf16_round(rng.standard_normal((128, 128)))
    enc = make_encoder(128, 128, torch.bfloat16, W)
    c = enc.compute_hash(x.cuda())
    assert tuple(c.shape) == (3, 5, 16)
    cn = enc.compute_hash((-x).cuda())
    assert torch.equal(cn, ~c)  # no projection is exactly zero for Gaussian data


def test_zero_and_nan_rows_give_zero_bits():
    enc = make_encoder(128, 128, torch.bfloat16, torch.eye(128))
    x = torch.zeros(2, 128)
    x[1, 2] = float("nan")
    x[1, 5] = 1.0
    c = enc.compute_hash(x.to(torch.bfloat16).cuda()).cpu().numpy()
    assert not c.any()


def test_per_head_weights_gqa_queries():
    """BASELINE.json config 2 query side: 32 q heads, one projection per KV head (group of 4)."""
    rng = rng_for(8)
    B, Hq, Hkv, K, N = 6, 32, 8, 128, 128
    x = bf16_round(rng.standard_normal((B, Hq, K)))
    W = bf16_round(rng.standard_normal((Hkv, K, N)))
    enc = make_encoder(K, N, torch.bfloat16, W, n_w=Hkv, hpw=Hq // Hkv)
    c = enc.compute_hash(x.cuda(), per_head=True).cpu().numpy()
    assert c.shape == (B, Hq, N // 8)
    for h in range(Hq):
        assert_codes_match(c[:, h], x[:, h].float().numpy(), W[h // 4].float().numpy())


@pytest.mark.parametrize("B,H,K,N,n_w", [
    (16, 64, 512, 512, 1),   # the latent-attention step's queries: 32 tiles of (token, head) pairs instead of 64 half-empty ones
    (3, 5, 128, 128, 1),     # 15 pairs: one partial tile
    (33, 3, 64, 64, 1),      # 99 pairs in 4 tiles against 2 x 3 by head
    (7, 6, 256, 256, 1),
    (40, 4, 128, 128, 1),    # 2 x 4 tiles by head, 5 by pair
    (7, 6, 128, 128, 2),     # two projections (3 heads each): tiles stay with one head
])
def test_few_tokens_many_heads_one_projection(B, H, K, N, n_w):
    """Rows of the small-row kernel's tiles are (token, head) pairs when one projection serves every
    head and that needs fewer tiles; the codes, and where they go (dense and through a slot mapping),
    are the same as head by head."""
    rng = rng_for(80 + B + H)
    x = bf16_round(rng.standard_normal((B, H, K)))
    W = bf16_round(rng.standard_normal((n_w, K, N)))
    hpw = H // n_w
    enc = make_encoder(K, N, torch.bfloat16, W, n_w=n_w, hpw=hpw)
    c = enc.compute_hash(x.cuda(), per_head=True).cpu().numpy()
    assert c.shape == (B, H, N // 8)
    for h in range(H):
        assert_codes_match(c[:, h], x[:, h].float().numpy(), W[h // hpw].float().numpy())
    # the same rows through the paged store, two dropped
    NB, BS = 5, 16
    slots = rng.permutation(NB * BS)[:B].astype(np.int64)
    slots[0] = -1
    if B > 2:
        slots[2] = NB * BS + 3
    cache = torch.full((NB, BS, H, N // 8), 0xAB, dtype=torch.uint8, device="cuda")
    enc.compute_hash_and_cache(x.cuda(), torch.from_numpy(slots).cuda(), cache, block_size=BS)
    expect = np.full((NB, BS, H, N // 32), 0xABABABAB, np.uint32)
    c_api.code_scatter(np.ascontiguousarray(c).view(np.uint32), slots, expect, BS)
    assert np.array_equal(cache.cpu().numpy().view(np.uint32), expect)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,K,N,n_w", [
    (224, 1, 512, 512, 1), (225, 1, 512, 512, 1), (256, 1, 256, 128, 1),  # seven row tiles, eight
    (8, 33, 512, 64, 1), (16, 33, 256, 96, 1),   # nine and seventeen row tiles of pairs; columns no power of two
    (40, 8, 512, 128, 8), (5, 12, 256, 64, 4),   # a projection per head or per three heads: two row tiles each, one
    (1, 1, 512, 512, 1), (21, 1, 512, 96, 1), (22, 1, 512, 512, 1), (3, 7, 512, 64, 1), (21, 8, 512, 128, 8),  # few rows in a tile
    (1, 3, 256, 96, 3), (27, 1, 256, 128, 1), (28, 1, 256, 64, 1), (2, 14, 256, 128, 1),
])
def test_split_row_tiles(dtype, B, H, K, N, n_w):
    """Rows of 256 and 512 values, few enough for the kernel whose waves share a row tile: both ways of reading the
    rows, the order in which row and column tiles go out, rows past the last, rows that lie apart (a strided view)."""
    rng = rng_for(B * 131 + H * 7 + K + N)
    wide = torch.from_numpy(rng.standard_normal((B, H, K + 24)).astype(np.float32)).to(dtype)
    W = torch.from_numpy(rng.standard_normal((n_w, K, N)).astype(np.float32)).to(dtype)
    enc = make_encoder(K, N, dtype, W if n_w > 1 else W[0], n_w=n_w, hpw=H // n_w)
    codes = enc.compute_hash(wide.cuda()[..., 8:8 + K], per_head=True).cpu().numpy()
    assert _encode_route(K, N, H, B).startswith("encode_small")
    x = wide[..., 8:8 + K].float().numpy()
    for h in range(H):
        assert_codes_match(codes[:, h], x[:, h], W[h // (H // n_w)].float().numpy())


@pytest.mark.parametrize("T,N,H,BS,dtype,route", [
    (1285, 512, 1, 64, torch.float16, "2,4"),    # eleven row tiles: three of the second eight streams; one row past a group of four
    (4097, 128, 3, 48, torch.bfloat16, "2,4"),   # heads side by side, block size no power of two, a last tile of one row
    (8063, 512, 1, 64, torch.bfloat16, "4,4"),   # 63 row tiles, one row short
    (20000, 384, 1, 64, torch.float16, "4,8"),   # streams that eight does not divide, a second tile for some
    (50001, 512, 1, 64, torch.bfloat16, "8,8"),  # a second row tile for some of the streams, the last one of a few rows
    (65535, 512, 1, 32, torch.bfloat16, "8,8"),  # two for all, one row short
    (545, 512, 1, 32, torch.bfloat16, "2,4"),    # the fewest rows: five row tiles, the last of one row
    (289, 1024, 1, 64, torch.float16, "2,4"),    # three
    # streams that eight does not divide, dealt out with their slices over all heads
    (1500, 384, 6, 64, torch.bfloat16, "4,4"),   # twelve, a tile each
    (3001, 384, 6, 48, torch.float16, "4,8"),    # twelve, the last tile of some rows
    (4609, 640, 4, 64, torch.bfloat16, "4,8"),   # twelve, a second tile for most, the last one of one row
    (2305, 640, 8, 64, torch.bfloat16, "4,8"),   # six, two tiles for most
    (1153, 384, 16, 64, torch.float16, "4,8"),   # five, a tile each, more heads
])
def test_rows_of_512_values_by_tile_shape(T, N, H, BS, dtype, route):
    """Every shape of the tile; one or several row tiles per workgroup; a strided view of the rows, rows that are
    skipped, zero or NaN.  The rows checked are those around tile edges and a sample of the others."""
    assert _encode_route(512, N, H, T) == "encode_pipe<%s>" % route
    rng = rng_for(T + N + H)
    g = torch.Generator(device="cuda")
    g.manual_seed(T)
    x = torch.randn(T, H, 512 + 8, generator=g, device="cuda", dtype=torch.float32).to(dtype)[..., 8:]
    x[T // 3] = 0.0
    x[T // 2, :, 5] = float("nan")
    W = torch.from_numpy(rng.standard_normal((512, N)).astype(np.float32)).to(dtype)
    enc = make_encoder(512, N, dtype, W)
    nb = -(-T // BS)
    ids = rng.permutation(nb)
    slot = ids[np.arange(T) // BS].astype(np.int64) * BS + np.arange(T) % BS
    stored = slot.copy()
    stored[7::11] = -1
    cache = torch.zeros((nb, BS, H, N // 32), dtype=torch.int32, device="cuda")
    enc.compute_hash_and_cache(x, torch.from_numpy(stored).cuda(), cache, block_size=BS)
    flat = cache.cpu().numpy().reshape(nb * BS, H, N // 32)
    assert not flat[slot[7::11]].any() and not flat[slot[[T // 3, T // 2]]].any()
    near = (np.arange(0, T + 128, 128)[:, None] + np.array([-33, -1, 0, 31, 32, 64])).reshape(-1)
    rows = np.unique(np.concatenate([near, [T - 2, T - 1], rng.integers(0, T, 2000)]))
    rows = rows[(rows >= 0) & (rows < T)]
    rows = rows[(stored[rows] >= 0) & (rows != T // 2)]
    xs = x[torch.from_numpy(rows).cuda()].float().cpu().numpy()
    for h in range(H):
        assert_codes_match(np.ascontiguousarray(flat[slot[rows], h]).view(np.uint8), xs[:, h], W.float().numpy())


@pytest.mark.parametrize("D,H,BS,T,dtype", [
    (128, 1, 32, 1, torch.bfloat16), (128, 8, 128, 130, torch.bfloat16), (64, 3, 96, 1000, torch.float16),
    (128, 3, 32, 8001, torch.float16), (64, 8, 64, 17000, torch.bfloat16),   # one tile a wave, two for some
    (128, 2, 128, 200001, torch.bfloat16),                                    # several tiles a wave, waves side by side
    (128, 8, 128, 530000, torch.bfloat16),                                    # more than the 64 whose blocks a wave holds
])
def test_rehash_of_rows_side_by_side(D, H, BS, T, dtype):
    """The streaming rehash: block ids outside the cache, a last block part full, zero and NaN rows, an untouched
    rest of the code cache.  Rows checked are the first, the last and a sample."""
    from ucm_amd import _lib

    g = torch.Generator(device="cuda")
    g.manual_seed(T + D)
    nb = -(-T // BS)
    kv = torch.randn(nb + 1, BS, H, D, generator=g, device="cuda", dtype=dtype)
    W = torch.from_numpy(rng_for(D + T).standard_normal((D, D)).astype(np.float32)).to(dtype)
    ids = torch.randperm(nb + 1, generator=g, device="cuda")[:nb].to(torch.int32)
    used = ids.cpu().numpy().copy()
    if nb > 5:
        ids[2], ids[4] = -1, nb + 1
        used[[2, 4]] = -1
        kv[int(used[1]), 1] = 0.0
        kv[int(used[1]), 2, :, 3] = float("nan")
    enc = make_encoder(D, D, dtype, W)
    fill = 0x55AA55AA
    cache = torch.full((nb + 1, BS, H, D // 32), fill, dtype=torch.int32, device="cuda")
    enc.compute_hash_from_paged_cache(kv, ids, T, cache, block_size=BS)
    assert _lib.last_encode() == "encode_run<%d,1>" % D
    t = np.unique(np.concatenate([np.arange(min(T, 300)), [T - 1, T - min(T, 40)], rng_for(T).integers(0, T, 3000)]))
    t = t[used[t // BS] >= 0]
    blk, tok = used[t // BS], t % BS
    b_t, k_t = torch.from_numpy(blk).long().cuda(), torch.from_numpy(tok).cuda()
    got, x = cache[b_t, k_t].cpu().numpy(), kv[b_t, k_t].float().cpu().numpy()
    nan = np.isnan(x).any(axis=(1, 2))
    assert not got[nan].any()
    for h in range(H):
        assert_codes_match(np.ascontiguousarray(got[~nan, h]).view(np.uint8), x[~nan, h], W.float().numpy())
    untouched = torch.ones(nb + 1, BS, dtype=torch.bool, device="cuda")
    full = torch.from_numpy(used[:nb - 1][used[:nb - 1] >= 0]).long().cuda()
    untouched[full] = False
    if used[nb - 1] >= 0:
        untouched[int(used[nb - 1]), :T - (nb - 1) * BS] = False
    assert (cache[untouched] == fill).all()


@pytest.mark.parametrize("D,H,T,slots,side,route", [
    (128, 8, 1301, "i64", 0, "encode_run<128,0>"), (128, 3, 9001, "i32", 0, "encode_run<128,0>"),  # rows that 32 does not divide
    (64, 1, 30001, "i64", 1, "encode_run<64,0>"),    # codes that are not aligned
    (128, 1, 65536, "dense", 0, "encode_run<128,0>"), (128, 1, 65537, "i64", 0, "encode_mfma<4,1,1>"),  # a tile to every wave, one more
])
def test_rows_side_by_side_by_slot(D, H, T, slots, side, route):
    from ucm_amd import _lib

    BS = 48
    g = torch.Generator(device="cuda")
    g.manual_seed(T + D)
    x = torch.randn(T, H, D, generator=g, device="cuda", dtype=torch.bfloat16)
    W = torch.from_numpy(rng_for(D + T).standard_normal((D, D)).astype(np.float32)).to(torch.bfloat16)
    enc = make_encoder(D, D, torch.bfloat16, W)
    nb = -(-T // BS)
    slot = rng_for(T).permutation(nb * BS)[:T].astype(np.int64)
    if slots == "dense":
        got = enc.compute_hash(x, per_head=True).cpu().numpy().reshape(T, H, D // 8)
        slot[:] = 0
    else:
        slot[5::9] = -1
        cache = torch.zeros((nb, BS, H, D // 32 + side), dtype=torch.int32, device="cuda")
        enc.compute_hash_and_cache(x, torch.from_numpy(slot).to(torch.int64 if slots == "i64" else torch.int32).cuda(),
                                   cache[..., side:], block_size=BS)
        flat = cache.cpu().numpy().reshape(nb * BS, H, D // 32 + side)
        assert not flat[np.setdiff1d(np.arange(nb * BS), slot)].any() and not flat[..., :side].any()
        got = np.ascontiguousarray(flat[np.maximum(slot, 0)][..., side:]).view(np.uint8)
    assert _lib.last_encode() == route
    keep = np.flatnonzero(slot >= 0)
    keep = np.unique(np.concatenate([keep[:500], keep[-100:], rng_for(T + 1).choice(keep, 2000)]))
    xs = x.float().cpu().numpy()[keep]
    for h in range(H):
        assert_codes_match(np.ascontiguousarray(got[keep, h]), xs[:, h], W.float().numpy())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("slot_dtype", [torch.int32, torch.int64])
def test_compute_hash_and_cache(dtype, slot_dtype):
    rng = rng_for(9)
    T, H, K, N, NB, BS = 200, 8, 128, 128, 6, 128
    x = torch.from_numpy(rng.standard_normal((T, H, K)).astype(np.float32)).to(dtype)
    W = torch.from_numpy(rng.standard_normal((H, K, N)).astype(np.float32)).to(dtype)
    slots = rng.permutation(NB * BS)[:T].astype(np.int64)
    slots[5] = -1
    slots[17] = NB * BS          # first slot past the cache
    slots[40] = NB * BS + 1000
    enc = make_encoder(K, N, dtype, W, n_w=H, hpw=1)
    cache = torch.full((NB, BS, H, N // 8), 0xAB, dtype=torch.uint8, device="cuda")
    out = enc.compute_hash_and_cache(x.cuda(), torch.from_numpy(slots).to(slot_dtype).cuda(),
                                     cache, block_size=BS)
    assert out is cache
    got = cache.cpu().numpy()
    # fused write == separate encode + the oracle's scatter (hash_encoder.py:136-195)
    codes = enc.compute_hash(x.cuda(), per_head=True).cpu().numpy()  # [T,H,16]
    expect = np.full((NB, BS, H, N // 32), 0xABABABAB, np.uint32)
    c_api.code_scatter(np.ascontiguousarray(codes).view(np.uint32), slots, expect, BS)
    assert np.array_equal(got.view(np.uint32), expect)
    for h in range(H):
        assert_codes_match(codes[:, h], x[:, h].float().numpy(), W[h].float().numpy())


# Row counts above 256 per head take the tiled MFMA kernel; the shapes below reach each of its
# compile-time variants: column tiles per group 4/2/1, unrolled and run-time group counts,
# the pipelined path (K <= 128) and the line-by-line path (K >= 256), partial last tiles and
# workgroups whose run of tiles ends past the tensor.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(257, 128, 128), (515, 128, 128), (1000, 128, 256), (4100, 128, 128),
                                   (700, 128, 512), (300, 128, 192), (300, 128, 96), (640, 128, 64),
                                   (385, 128, 32), (513, 64, 64), (900, 64, 128), (300, 64, 32),
                                   (600, 256, 128), (300, 512, 256), (2049, 512, 128)])
def test_tiled_kernel_shapes(dtype, M, K, N):
    rng = rng_for(2000 + M + K + N)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dtype)
    W = torch.from_numpy(rng.standard_normal((K, N)).astype(np.float32)).to(dtype)
    enc = make_encoder(K, N, dtype, W)
    codes = enc.compute_hash(x.cuda())
    assert tuple(codes.shape) == (M, N // 8)
    assert_codes_match(codes.cpu().numpy(), x.float().numpy(), W.float().numpy())


@pytest.mark.parametrize("slot_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("T,H,BS", [(700, 8, 128), (1029, 4, 48), (300, 2, 16)])
def test_tiled_kernel_paged_store(slot_dtype, T, H, BS):
    """Fused cache write of the tiled kernel: permuted and invalid slots, a block size that is
    not a power of two, head-interleaved input rows, cells outside the slots untouched."""
    rng = rng_for(12 + T)
    K = N = 128
    NB = (T + BS - 1) // BS + 3
    x = bf16_round(rng.standard_normal((T, H, K)))
    W = bf16_round(rng.standard_normal((H, K, N)))
    slots = rng.permutation(NB * BS)[:T].astype(np.int64)
    slots[3] = -1
    slots[T // 2] = NB * BS
    slots[T - 1] = NB * BS + 77
    enc = make_encoder(K, N, torch.bfloat16, W, n_w=H, hpw=1)
    cache = torch.full((NB, BS, H, N // 8), 0xAB, dtype=torch.uint8, device="cuda")
    enc.compute_hash_and_cache(x.cuda(), torch.from_numpy(slots).to(slot_dtype).cuda(), cache,
                               block_size=BS)
    codes = np.stack([brute.hash_encode(x[:, h].float().numpy(), W[h].float().numpy())
                      for h in range(H)], axis=1)  # [T,H,4] uint32
    expect = np.full((NB, BS, H, N // 32), 0xABABABAB, np.uint32)
    c_api.code_scatter(np.ascontiguousarray(codes), slots, expect, BS)
    got = cache.cpu().numpy().view(np.uint32)
    if not np.array_equal(got, expect):
        # differences may only be margin bits of rows that were written
        gpu_codes = enc.compute_hash(x.cuda(), per_head=True).cpu().numpy()
        for h in range(H):
            assert_codes_match(gpu_codes[:, h], x[:, h].float().numpy(), W[h].float().numpy())
        expect2 = np.full((NB, BS, H, N // 32), 0xABABABAB, np.uint32)
        c_api.code_scatter(np.ascontiguousarray(gpu_codes).view(np.uint32), slots, expect2, BS)
        assert np.array_equal(got, expect2)


def test_tiled_kernel_strided_rows_and_dense_heads():
    """Rows that are a slice of a wider tensor (row pitch 3*K) and a dense per-head output."""
    rng = rng_for(13)
    T, H, K, N = 520, 3, 128, 128
    wide = bf16_round(rng.standard_normal((T, H, 3 * K))).cuda()
    x = wide[:, :, K:2 * K]
    W = bf16_round(rng.standard_normal((K, N)))
    enc = make_encoder(K, N, torch.bfloat16, W)
    c = enc.compute_hash(x, per_head=True).cpu().numpy()  # keeps the row pitch; one matrix
    assert c.shape == (T, H, N // 8)
    xs = x.float().cpu().numpy()
    for h in range(H):
        assert_codes_match(c[:, h], xs[:, h], W.float().numpy())


@pytest.mark.parametrize("dtype,BS,H,n_blocks,n_tokens,per_head", [
    (torch.bfloat16, 128, 8, 9, 1100, True),    # tiled kernel, partial last block
    (torch.float16, 128, 2, 40, 5120, False),   # several workgroups per head
    (torch.bfloat16, 64, 4, 3, 130, False),     # few rows: latency kernel
    (torch.bfloat16, 32, 4, 20, 640, True),     # a wave per block
    (torch.bfloat16, 48, 2, 12, 570, False),    # block size not a multiple of 32: FMA kernel
    (torch.float32, 16, 2, 5, 77, False),       # fp32: FMA kernel
])
def test_rehash_from_paged_cache(dtype, BS, H, n_blocks, n_tokens, per_head):
    """Prefix-cache rehash against the CPU checker and against the reference's own recipe run
    on the GPU (gather the blocks, then compute_hash_and_cache with the prefix slot mapping)."""
    rng = rng_for(300 + BS + n_blocks)
    K = N = 128
    NBk, NB = n_blocks + 6, n_blocks + 4
    kc = torch.from_numpy(rng.standard_normal((NBk, BS, H, K)).astype(np.float32)).to(dtype)
    W = torch.from_numpy(rng.standard_normal((H if per_head else 1, K, N)).astype(np.float32)).to(dtype)
    ids = rng.permutation(NB)[:n_blocks].astype(np.int32)
    if n_blocks >= 5:
        ids[1] = -1            # unusable entries drop their tokens
        ids[3] = NB + 1        # valid in the KV cache, outside the code cache
    enc = make_encoder(K, N, dtype, W if per_head else W[0], n_w=H if per_head else 1, hpw=1)
    cache = torch.full((NB, BS, H, N // 8), 0xAB, dtype=torch.uint8, device="cuda")
    out = enc.compute_hash_from_paged_cache(kc.cuda(), torch.from_numpy(ids).cuda(), n_tokens, cache,
                                            block_size=BS)
    assert out is cache
    got = cache.cpu().numpy().view(np.uint32)

    # the reference's recipe on the GPU: gather, slot mapping, fused encode + store
    cache2 = torch.full_like(cache, 0xAB)
    tok = np.arange(n_tokens)
    slots = ids[tok // BS].astype(np.int64) * BS + tok % BS
    slots[(ids[tok // BS] < 0) | (ids[tok // BS] >= NB)] = -1
    gathered = kc.cuda()[torch.from_numpy(np.clip(ids, 0, NBk - 1)).long().cuda()].reshape(-1, H, K)[:n_tokens]
    enc.compute_hash_and_cache(gathered.contiguous(), torch.from_numpy(slots).cuda(), cache2, block_size=BS)
    assert torch.equal(cache, cache2)

    # CPU checker (bits may differ only inside the margin)
    expect = np.full((NB, BS, H, N // 32), 0xABABABAB, np.uint32)
    c_api.hash_encode_paged(kc.float().numpy(), ids, n_tokens, W.float().numpy(),
                            1 if per_head else 0, expect)
    if not np.array_equal(got, expect):
        kcn, Wn = kc.float().numpy(), W.float().numpy()
        for i in range(n_tokens):
            b = int(ids[i // BS])
            if b < 0 or b >= NB:
                continue
            for h in range(H):
                assert_codes_match(got[b, i % BS, h:h + 1].view(np.uint8),
                                   kcn[b, i % BS, h:h + 1], Wn[h if per_head else 0])
    # cells of skipped and unlisted blocks stay untouched
    listed = {int(b) for b in ids if 0 <= b < NB}
    for b in range(NB):
        if b not in listed:
            assert (got[b] == 0xABABABAB).all()


def test_rehash_argument_errors():
    enc = make_encoder(128, 128, torch.bfloat16, torch.eye(128))
    kc = torch.zeros((4, 64, 2, 128), dtype=torch.bfloat16, device="cuda")
    cache = torch.zeros((4, 64, 2, 16), dtype=torch.uint8, device="cuda")
    ids = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        enc.compute_hash_from_paged_cache(kc, ids, 129, cache, block_size=64)   # > 2 blocks
    with pytest.raises(ValueError):
        enc.compute_hash_from_paged_cache(kc, ids.long(), 10, cache, block_size=64)
    with pytest.raises(ValueError):
        enc.compute_hash_from_paged_cache(kc, ids, 10, cache, block_size=128)
    with pytest.raises(ValueError):
        enc.compute_hash_from_paged_cache(kc.float(), ids, 10, cache, block_size=64)
    assert enc.compute_hash_from_paged_cache(kc, ids, 0, cache, block_size=64) is cache


def test_cache_as_bf16_view_and_shared_weight():
    """The plugin allocates the code cache as bfloat16 [NB,BS,H,hash_numbers/2]
    (hash_encoder.py:509-546) and uses one projection for all heads."""
    rng = rng_for(10)
    T, H, K, N, NB, BS = 64, 4, 128, 128, 2, 64
    x = bf16_round(rng.standard_normal((T, H, K)))
    W = bf16_round(rng.standard_normal((K, N)))
    enc = make_encoder(K, N, torch.bfloat16, W)
    cache = torch.zeros((NB, BS, H, N // 16), dtype=torch.bfloat16, device="cuda")
    slots = torch.arange(T, dtype=torch.int64, device="cuda") + 10
    enc.compute_hash_and_cache(x.cuda(), slots, cache, block_size=BS)
    got = cache.view(torch.uint8).cpu().numpy().reshape(NB * BS, H, N // 8)
    for h in range(H):
        assert_codes_match(got[10:10 + T, h], x[:, h].float().numpy(), W.float().numpy())
    assert not got[:10].any() and not got[10 + T:].any()


def test_reshape_and_cache_head_major_shape_of_the_reference_fixture():
    """Shapes of ucm/sparse/test/gsa/pt/npu_reshape_and_cache_bnsd_tensor.pt (that file holds
    inputs only): 1 token, 2 heads, 16-byte codes, slot 22552, head-major cache
    [402, 2, 128, 16].  Data here is synthetic."""
    from ucm_amd.sparse.hash_encoder import reshape_and_cache_khash

    rng = rng_for(11)
    codes = torch.from_numpy(rng.integers(0, 256, size=(1, 2, 16), dtype=np.uint8)).cuda()
    cache_hm = torch.zeros((402, 2, 128, 16), dtype=torch.uint8, device="cuda")
    slot = torch.tensor([22552], dtype=torch.int32, device="cuda")
    # token-major view [NB, BS, H, W] of the head-major storage
    reshape_and_cache_khash(codes, slot, cache_hm.permute(0, 2, 1, 3), block_size=128)
    got = cache_hm.cpu().numpy()
    assert np.array_equal(got[176, :, 24, :], codes[0].cpu().numpy())
    got[176, :, 24, :] = 0
    assert not got.any()


def test_argument_errors_match_the_reference_behaviour():
    from ucm_amd.sparse import HashEncoder

    with pytest.raises(ValueError):
        HashEncoder(128, 100, torch.bfloat16, torch.device("cuda:0"))
    enc = HashEncoder(128, 128, torch.bfloat16, torch.device("cuda:0"))
    with pytest.raises(ValueError):
        enc.compute_hash(torch.zeros(4, 64, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(ValueError):
        enc.compute_hash(torch.zeros(4, 128, dtype=torch.bfloat16))  # wrong device
    with pytest.raises(ValueError):
        enc.set_hash_weight(torch.zeros(128, 64, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(ValueError):
        enc.set_hash_weight(torch.zeros(128, 128, dtype=torch.float32, device="cuda"))
    cache = torch.zeros((2, 64, 4, 16), dtype=torch.uint8, device="cuda")
    x = torch.zeros(3, 4, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError):
        enc.compute_hash_and_cache(x, torch.zeros(2, dtype=torch.int64, device="cuda"), cache, 64)
    with pytest.raises(ValueError):
        enc.compute_hash_and_cache(x, torch.zeros(3, dtype=torch.int64, device="cuda"), cache, 128)
    # Haar-orthogonal default weights: W^T W = I
    w = enc.hash_weights.float()
    assert torch.allclose(w.T @ w, torch.eye(128, device="cuda"), atol=5e-2)


def test_unpack_hash_roundtrip():
    enc = make_encoder(128, 128, torch.bfloat16, torch.eye(128))
    x = torch.zeros(2, 128)
    x[0, 3] = 1.0
    x[1, 100] = 1.0
    c = enc.compute_hash(x.to(torch.bfloat16).cuda())
    pm = enc._unpack_hash(c).cpu()
    assert pm[0, 3] == 1 and pm[1, 100] == 1 and pm.sum() == 2 - (256 - 2)


@pytest.mark.parametrize("T,N,H,n_w,slots", [
    (1281, 512, 1, 1, "i64"),    # 32-column slices, a last tile of one row
    (2049, 512, 1, 1, "i32"),    # 64-column slices
    (4097, 512, 1, 1, "i64"),    # 128-column slices, one tile per workgroup
    (8321, 512, 1, 1, "paged"),  # the same, a second tile for some
    (2300, 256, 2, 2, "paged"),  # a projection per head
    (30000, 96, 1, 1, "i32"),    # column count only 32 divides, several tiles per workgroup
    (30001, 192, 1, 1, "dense"), # ... only 64 divides
    (70001, 96, 1, 1, "paged"),  # past the slices: four row tiles a workgroup, 96-column and
    (17000, 224, 1, 1, "i64"),   # 32-column slices
    (60001, 192, 1, 1, "dense"),
    (3000, 320, 2, 1, "i64"),
])
def test_rows_of_512_values_at_the_edges_of_slices_and_tiles(T, N, H, n_w, slots):
    """One instantiation per slice width; one or several row tiles per workgroup; rows that do not exist,
    are skipped or hold NaN."""
    rng = rng_for(T + N + H)
    K, BS = 512, 64
    x32 = rng.standard_normal((T, H, K)).astype(np.float32)
    x32[T // 3] = 0.0
    x32[T // 2, :, 5] = np.nan
    x = torch.from_numpy(x32).to(torch.bfloat16)
    W = torch.from_numpy(rng.standard_normal((n_w, K, N)).astype(np.float32)).to(torch.bfloat16)
    enc = make_encoder(K, N, torch.bfloat16, W if n_w > 1 else W[0], n_w=n_w, hpw=1)
    nb = -(-T // BS)
    ids = rng.permutation(nb).astype(np.int32)
    slot = ids[np.arange(T) // BS].astype(np.int64) * BS + np.arange(T) % BS
    cache = torch.zeros((nb, BS, H, N // 32 + 1), dtype=torch.int32, device="cuda")  # rows of other codes between
    view = cache[..., 1:]
    if slots == "paged":
        kv = torch.zeros((nb * BS, H, K), dtype=torch.bfloat16)
        kv[torch.from_numpy(slot)] = x
        enc.compute_hash_from_paged_cache(kv.view(nb, BS, H, K).cuda(), torch.from_numpy(ids).cuda(), T, view, block_size=BS)
    elif slots == "dense":
        got = enc.compute_hash(x.cuda(), per_head=True).cpu().numpy().reshape(T, H, N // 8)
    else:
        slot[7::11] = -1  # rows that are skipped
        enc.compute_hash_and_cache(x.cuda(), torch.from_numpy(slot).to(torch.int64 if slots == "i64" else torch.int32).cuda(),
                                   view, block_size=BS)
    if slots != "dense":
        flat = cache.cpu().numpy().reshape(nb * BS, H, N // 32 + 1)
        assert not flat[:, :, 0].any()
        unused = np.setdiff1d(np.arange(nb * BS), slot)
        assert not flat[unused].any()
        got = np.ascontiguousarray(flat[np.maximum(slot, 0)][:, :, 1:]).view(np.uint8)
    keep = np.flatnonzero(slot >= 0)
    nan = keep[keep == T // 2]
    assert not got[nan].any() and not got[keep[keep == T // 3]].any()  # NaN > 0 and 0 > 0 are false
    rows = keep[keep != T // 2]
    for h in range(H):
        assert_codes_match(got[rows, h], x[rows, h].float().numpy(), W[min(h, n_w - 1)].float().numpy())


@pytest.mark.parametrize("K,N,H,T,paged", [
    (128, 128, 8, 1025, True),    # one row tile per workgroup, the last with one row
    (128, 128, 2, 6001, False),
    (64, 64, 8, 1500, True),
    (64, 128, 4, 24600, False),   # just past three workgroups a compute unit: four tiles each
    (128, 128, 8, 12500, True),
    (128, 256, 1, 98400, False),
    (128, 128, 8, 65700, True),   # eight tiles each
    (64, 128, 8, 65700, True),    # ... of 64 values
    (64, 64, 8, 10300, False),    # the streaming kernel's first sizes at 64 x 64
])
def test_row_tiles_per_workgroup(K, N, H, T, paged):
    """One instantiation per number of row tiles a workgroup encodes, at the edges of their ranges; a sample
    of rows (the first, the last, every tile position) against the oracle."""
    rng = rng_for(T + N)
    BS, nb = 64, -(-T // 64)
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(nb * BS, H, K, generator=g, device="cuda").to(torch.bfloat16)
    W = torch.from_numpy(rng.standard_normal((K, N)).astype(np.float32)).to(torch.bfloat16)
    enc = make_encoder(K, N, torch.bfloat16, W)
    ids = torch.from_numpy(rng.permutation(nb).astype(np.int32)).cuda()
    cache = torch.zeros((nb, BS, H, N // 32), dtype=torch.int32, device="cuda")
    t = torch.arange(T, device="cuda")
    slot = ids[t // BS].long() * BS + t % BS
    if paged:
        enc.compute_hash_from_paged_cache(x.view(nb, BS, H, K), ids, T, cache, block_size=BS)
        x = x[slot]
    else:
        enc.compute_hash_and_cache(x[:T], slot, cache, block_size=BS)
    flat = cache.view(nb * BS, H, N // 32)
    rest = torch.ones(nb * BS, dtype=torch.bool, device="cuda")
    rest[slot] = False
    assert not flat[rest].any()
    rows = np.unique(np.concatenate([np.arange(130), T - 1 - np.arange(130), rng.integers(0, T, 1500)]))
    pick = torch.from_numpy(rows).cuda()
    got = flat[slot[pick]].cpu().numpy().view(np.uint8)
    xs = x[pick].float().cpu().numpy()
    for h in range(H):
        assert_codes_match(got[:, h], xs[:, h], W.float().numpy())


@pytest.mark.parametrize("K,N,H,T,paged,route", [
    (128, 128, 8, 1025, True, "4,1,1"), (128, 128, 8, 12500, True, "4,1,4"), (128, 128, 8, 65700, True, "4,1,8"),
    (64, 64, 8, 10001, True, "2,1,1"), (64, 64, 4, 20001, True, "2,1,1"),
    (128, 128, 8, 8193, False, "4,1,1"), (128, 128, 8, 12400, False, "4,1,4"), (128, 128, 8, 65700, False, "4,1,8"),
    (64, 64, 8, 9001, False, "2,1,1"), (64, 128, 8, 65700, False, "4,1,8"), (128, 256, 1, 66000, False, "4,2,4"),
])
def test_row_tiles_of_the_tiled_kernel(K, N, H, T, paged, route):
    """The codes of each number of row tiles where that kernel is the one that runs: by slot beyond a tile a wave of the
    streaming one, paged inputs whose rows lie apart."""
    from ucm_amd import _lib

    rng = rng_for(T * 3 + N)
    BS, nb = 64, -(-T // 64)
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(nb * BS, H, K + 8, generator=g, device="cuda").to(torch.bfloat16)[..., 8:]
    W = torch.from_numpy(rng.standard_normal((K, N)).astype(np.float32)).to(torch.bfloat16)
    enc = make_encoder(K, N, torch.bfloat16, W)
    ids = torch.from_numpy(rng.permutation(nb).astype(np.int32)).cuda()
    cache = torch.zeros((nb, BS, H, N // 32), dtype=torch.int32, device="cuda")
    t = torch.arange(T, device="cuda")
    slot = ids[t // BS].long() * BS + t % BS
    if paged:
        enc.compute_hash_from_paged_cache(x.unflatten(0, (nb, BS)), ids, T, cache, block_size=BS)
        x = x[slot]
    else:
        x = x[:T].contiguous()
        enc.compute_hash_and_cache(x, slot, cache, block_size=BS)
    assert _lib.last_encode() == "encode_mfma<%s>" % route
    flat = cache.view(nb * BS, H, N // 32)
    rest = torch.ones(nb * BS, dtype=torch.bool, device="cuda")
    rest[slot] = False
    assert not flat[rest].any()
    rows = np.unique(np.concatenate([np.arange(130), T - 1 - np.arange(130), rng.integers(0, T, 1500)]))
    pick = torch.from_numpy(rows).cuda()
    got = flat[slot[pick]].cpu().numpy().view(np.uint8)
    xs = x[pick].float().cpu().numpy()
    for h in range(H):
        assert_codes_match(got[:, h], xs[:, h], W.float().numpy())


def _encode_route(K, N, H, T):
    """The kernel that a plain encode into a paged cache takes."""
    from ucm_amd import _lib

    enc = make_encoder(K, N, torch.bfloat16, torch.ones(K, N, dtype=torch.bfloat16))
    nb = -(-T // 64)
    cache = torch.zeros((nb, 64, H, N // 32), dtype=torch.int32, device="cuda")
    enc.compute_hash_and_cache(torch.ones(T, H, K, dtype=torch.bfloat16, device="cuda"), torch.arange(T, device="cuda"), cache,
                               block_size=64)
    return _lib.last_encode()


@pytest.mark.parametrize("K,N,T", [(64, 96, 1300), (64, 192, 1700), (64, 320, 1300), (64, 512, 800), (128, 96, 2200),
                                   (128, 160, 1000), (128, 192, 2200), (128, 224, 1700), (128, 384, 1300), (128, 512, 2500)])
def test_column_counts_without_a_one_tile_form_keep_the_small_kernel(K, N, T):
    """The tiled kernel has one row tile per workgroup for slices of 32, 64, 128 and 256 columns only; with four
    it took 1.3 to 2.9 times the small kernel's time at these sizes."""
    assert _encode_route(K, N, 8, T) == "encode_small"


@pytest.mark.parametrize("K,N,H,T,small", [
    (128, 128, 8, 700, True), (128, 128, 8, 1300, False), (128, 128, 1, 6000, True), (128, 128, 1, 12000, False),
    (128, 64, 8, 1000, True), (128, 64, 8, 1700, False), (128, 256, 8, 700, True), (128, 256, 8, 1300, False),
    (64, 128, 8, 1000, True), (64, 128, 8, 3000, False), (64, 64, 8, 1700, True), (64, 64, 8, 4000, False),
    (64, 32, 8, 6000, True), (128, 32, 8, 6000, False), (64, 256, 1, 5000, True), (64, 256, 8, 3000, False),
])
def test_small_kernel_up_to_where_the_tiled_one_is_as_fast(K, N, H, T, small):
    """Sizes on both sides of the equal times, some way off them."""
    assert (_encode_route(K, N, H, T) == "encode_small") == small


@pytest.mark.parametrize("N,H,T,small", [
    (512, 1, 448, True), (512, 1, 640, False), (512, 1, 1000, False), (256, 1, 960, True), (256, 1, 1200, False),
    (128, 1, 1900, True), (128, 1, 2500, False), (1024, 1, 224, True), (1024, 1, 300, False), (512, 8, 56, True), (512, 8, 90, False), (512, 32, 20, False),
    (512, 64, 16, True), (1024, 64, 8, True), (256, 128, 16, True),
    (192, 1, 1300, True), (192, 1, 4000, False), (64, 1, 8000, True),
])
def test_small_kernel_up_to_where_rows_of_512_values_stream(N, H, T, small):
    """A tile to a compute unit where the other kernel is the ring of chunks; more where it is the slices."""
    assert (_encode_route(512, N, H, T) == "encode_small") == small


@pytest.mark.parametrize("K,N,H,T,tiles", [
    (128, 128, 8, 12288, 1), (128, 128, 8, 12400, 4), (64, 128, 4, 24600, 4), (64, 64, 8, 10000, 1), (128, 256, 1, 65536, 1),
    (128, 256, 1, 66000, 4), (64, 256, 8, 12288, 1), (128, 128, 1, 98304, 1), (128, 128, 8, 65700, 8), (64, 32, 8, 65700, 8),
])
def test_row_tiles_per_workgroup_by_the_number_of_workgroups(K, N, H, T, tiles):
    """One row tile up to three workgroups a compute unit (two where a slice fills the LDS), eight from sixteen."""
    route = _encode_route(K, N, H, T)
    assert route.startswith("encode_mfma<") and route.endswith(",%d>" % tiles), route


@pytest.mark.parametrize("N,T,slices", [(96, 49152, True), (96, 70000, False), (160, 16384, True), (160, 24576, False), (192, 32768, True),
                                        (192, 60000, False), (192, 70000, True), (416, 8192, False), (288, 16384, True),
                                        (320, 65536, True), (32, 131072, True)])
def test_slices_of_512_values_up_to_where_they_read_the_rows_too_often(N, T, slices):
    route = _encode_route(512, N, 1, T)
    assert route.startswith("encode_slice<" if slices else "encode_mfma<"), route


@pytest.mark.parametrize("N,T,wide", [(256, 65535, False), (256, 65536, True), (512, 131071, False), (512, 131072, True)])
def test_rows_from_which_512_values_take_the_persistent_kernel(N, T, wide):
    assert (_encode_route(512, N, 1, T) == "encode_wide") == wide
