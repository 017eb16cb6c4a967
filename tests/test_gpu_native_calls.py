"""The native fronts (csrc/native_calls.cpp) against the general Python path of the same calls: same outputs
for what both take, the general path's answer for everything else."""
import contextlib

import pytest
import torch

from ucm_amd import _lib


class _NoFront:
    """Stands in for the module of fronts: every call is the general path's."""

    def __getattr__(self, name):
        return lambda *a: None


@contextlib.contextmanager
def general_path():
    real = _lib.native()
    _lib._native = _NoFront()
    try:
        yield
    finally:
        _lib._native = real


def test_fronts_leave_what_is_not_plain_to_the_general_path():
    n = _lib.native()
    t = torch.zeros(2, 2)
    assert n.dot_topk(t, t, t.int(), 1, None) is None  # not on a GPU
    for name in ("gsa_step", "sparse_step", "gsa_step_mla", "encode_cache", "encode_paged", "dot_topk", "kvstar_topk"):
        assert getattr(n, name)() is None and getattr(n, name)(*[object()] * 22) is None


# ---- one state per call; variant names a change that stays valid, takes the general path or is refused ----


def _encoder(din, bits, dtype):
    from ucm_amd.sparse import HashEncoder

    enc = HashEncoder(din, bits, dtype, torch.device("cuda:0"))
    g = torch.Generator(device="cuda").manual_seed(7)
    enc.set_hash_weight(torch.randn(din, bits, device="cuda", generator=g).to(dtype))
    return enc


def _randn(*s, dtype=torch.bfloat16, seed=1):
    return torch.randn(*s, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)).to(dtype)


def _strided(t):
    """The same values in every second row of a wider tensor."""
    wide = torch.zeros((2 * t.shape[0],) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
    wide[::2] = t
    return wide[::2]


def _encode(variant):
    x, slot = _randn(70, 4, 128), torch.randperm(3 * 32, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))[:70]
    cache = torch.zeros((3, 32, 4, 16), dtype=torch.uint8, device="cuda")
    if variant == "strided":
        x, slot = _strided(x), _strided(slot)
    elif variant == "one":  # extents of 1 with arbitrary strides
        x, slot = torch.as_strided(x, (1, 4, 128), (3, 128, 1)), slot[:1]
    elif variant == "wider_type":
        cache = cache.view(torch.int32)
    elif variant == "converted":
        x = x.float()
    elif variant == "wrong":
        slot = slot[:-1]
    enc = _encoder(128, 128, torch.bfloat16)
    return lambda: enc.compute_hash_and_cache(x, slot, cache, block_size=32).clone()


def _rehash(variant):
    kv, ids = _randn(5, 32, 2, 128), torch.tensor([3, 0, 4], dtype=torch.int32, device="cuda")
    cache = torch.zeros((5, 32, 2, 4), dtype=torch.int32, device="cuda")
    n = 96
    if variant == "strided":
        kv, ids = _strided(kv), _strided(ids)
    elif variant == "one":
        n = 1
    elif variant == "wrong":
        n = 97
    enc = _encoder(128, 128, torch.bfloat16)
    return lambda: enc.compute_hash_from_paged_cache(kv, ids, n, cache, block_size=32).clone()


def _paged(B, blocks, words):
    g = torch.Generator(device="cuda").manual_seed(5)
    cache = torch.randint(-2 ** 31, 2 ** 31, (B * blocks, 64) + words, dtype=torch.int32, device="cuda", generator=g)
    table = torch.randperm(B * blocks, device="cuda", generator=g).to(torch.int32).view(B, blocks)
    lens = torch.tensor([blocks * 64 - 5 * i for i in range(B)], dtype=torch.int32, device="cuda")
    return cache, table, lens, torch.arange(B, device="cuda") * 3


def _gqa(cls, variant):
    from ucm_amd.sparse import decode_step as D

    B, blocks = 3, 20
    cache, table, lens, slots = _paged(B, blocks, (2, 4))
    keys, q = _randn(B, 2, 128, seed=2), _randn(B, 8, 128, seed=3)
    if variant == "strided":
        keys, q, cache, table = _strided(keys), _strided(q), _strided(cache), _strided(table)
    elif variant == "one":
        keys, slots = torch.as_strided(keys, (1, 2, 128), (1, 128, 1)), slots[:1]
    elif variant == "wider_type":
        slots = slots.int()
    elif variant == "converted":
        keys = None
    elif variant == "wrong":
        lens = lens.long()
    w = _randn(128, 128, seed=4)
    step = (D.GSADecodeStep(w, 8, 2, B, blocks, 8 * 64, block_size=64) if cls == "gsa"
            else D.SparseDecodeStep(w, 8, 2, B, blocks, 8, block_size=64))
    return lambda: [t.clone() for t in (*step.step(keys, slots, q, cache, table, lens), cache)]


def _mla(variant):
    from ucm_amd.sparse import decode_step as D

    B, blocks = 2, 20
    cache, table, lens, slots = _paged(B, blocks, (18,))
    a = [_randn(B, 512, seed=2), _randn(B, 64, seed=3), slots, _randn(B, 8, 512, seed=4), _randn(B, 8, 64, seed=5), cache, table, lens]
    if variant == "strided":
        for i in (0, 1, 3, 4, 5, 6):
            a[i] = _strided(a[i])
    elif variant == "one":
        a[0], a[1], a[2] = torch.as_strided(a[0], (1, 512), (1, 1)), a[1][:1], slots[:1]
    elif variant == "wider_type":
        a[2] = slots.int()
    elif variant == "converted":
        a[0] = a[1] = a[2] = None
    elif variant == "wrong":
        a[3] = a[3].float()
    step = D.GSADecodeStepMLA(_randn(512, 512, seed=6), _randn(64, 64, seed=7), 8, 2, B, blocks, 8 * 64)
    return lambda: [t.clone() for t in (*step.step(*a), a[5])]


def _dot(variant):
    from ucm_amd.sparse.esa_retrieval_worker import dot_topk

    data, q = _randn(500, 64, dtype=torch.float32), _randn(2, 64, dtype=torch.float32, seed=2)
    idx = torch.randint(-1, 500, (2, 300), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).int()
    k, ws = 40, None
    if variant == "strided":
        data, q, idx = _strided(data), _strided(q), _strided(idx)
    elif variant == "one":
        data, idx = data[:1], torch.zeros_like(idx)
    elif variant == "wider_type":
        ws = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
    elif variant == "converted":
        idx = idx[:, :0]
    elif variant == "wrong":
        k = 5000  # more than the kernel orders
    return lambda: dot_topk(data, q, idx, k, ws)


def _kvstar(variant):
    from ucm_amd.sparse.kvstar_retrieve import kvstar_topk

    q, k = _randn(4, 8, 64, dtype=torch.float16), _randn(30, 8, 2, 32, dtype=torch.float16, seed=2)
    pr = torch.arange(0, 64, 2, device="cuda").repeat(2, 1)
    topk, ws = 10, None
    if variant == "strided":
        q, k, pr = _strided(q), _strided(k), _strided(pr)
    elif variant == "one":
        topk = 100
    elif variant == "wider_type":
        ws = torch.empty(1 << 22, dtype=torch.uint8, device="cuda")
    elif variant == "converted":
        pr = pr.cpu()
    elif variant == "wrong":
        pr = None
    return lambda: kvstar_topk(q, k, pr, topk, ws)


CALLS = {"encode": _encode, "rehash": _rehash, "gsa": lambda v: _gqa("gsa", v), "sparse": lambda v: _gqa("sparse", v),
         "mla": _mla, "dot": _dot, "kvstar": _kvstar}


def _outcome(make, variant):
    call = make(variant)
    try:
        out = call()
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)
    torch.cuda.synchronize()
    return [t.cpu() for t in (out if isinstance(out, (list, tuple)) else [out])]


@pytest.mark.gpu
@pytest.mark.parametrize("variant", ["plain", "strided", "one", "wider_type", "converted", "wrong", "side_stream"])
@pytest.mark.parametrize("name", list(CALLS))
def test_front_and_general_path_agree(name, variant):
    with general_path():
        want = _outcome(CALLS[name], variant)
    stream = torch.cuda.Stream() if variant == "side_stream" else torch.cuda.current_stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        got = _outcome(CALLS[name], variant)
    if variant == "wrong":
        assert isinstance(want, tuple) and got == want
        return
    assert not isinstance(want, tuple), want
    assert len(got) == len(want)
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and g.shape == w.shape and torch.equal(g, w)


def _tensors(call):
    for cell in call.__closure__:
        v = cell.cell_contents
        for t in v if isinstance(v, list) else [v]:
            if isinstance(t, torch.Tensor):
                yield t


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CALLS))
def test_fronts_issue_on_the_current_stream(name):
    """The inputs hold zeros until work that takes a few milliseconds has run on the current stream: a launch on
    any other stream would read those."""
    with general_path():
        want = _outcome(CALLS[name], "plain")
    call = CALLS[name]("plain")
    later = [(t, t.clone()) for t in _tensors(call)]
    assert len(later) >= 3
    for t, _ in later:
        t.zero_()
    busy = torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            busy = busy @ busy
            busy /= busy.abs().max()
        for t, good in later:
            t.copy_(good)
        out = call()
        assert not side.query()  # still busy: the call did not wait
    side.synchronize()
    for g, w in zip(out if isinstance(out, (list, tuple)) else [out], want):
        assert torch.equal(g.cpu(), w)


@pytest.mark.gpu
def test_plain_calls_take_the_front():
    calls = {n: m("plain") for n, m in CALLS.items()}

    class Spy:
        used = set()

        def __getattr__(self, name):
            def f(*a):
                r = getattr(real, name)(*a)
                if r is not None:
                    Spy.used.add(name)
                return r
            return f

    real = _lib.native()
    _lib._native = Spy()
    try:
        for c in calls.values():
            c()
    finally:
        _lib._native = real
    assert Spy.used == {"gsa_step", "sparse_step", "gsa_step_mla", "encode_cache", "encode_paged", "dot_topk", "kvstar_topk"}
