"""The calls a serving process makes into this library, as timed cases.

Eight kinds, each through the public entry point that a plugin or connector calls:

  gqa_decode  GSADecodeStep.step         per layer and decode step of a grouped-query model: new keys hashed
                                         into the paged code cache, mean query hashed, blocks scored, the
                                         replacement block table and lengths written
  gqa_topk    SparseDecodeStep.step      the same step with one list per KV head and its scores
  mla_decode  GSADecodeStepMLA.step      the decode step of a latent-attention model
  gqa_encode  compute_hash_and_cache     prefill: the codes of a chunk of keys, by slot
  mla_encode  compute_hash_and_cache x2  prefill of the latent part and the rope part of a code row
  rehash      compute_hash_from_paged_cache   a prefix loaded from the store is hashed where it lies
  esa         dot_topk                   float retrieval over block vectors
  kvstar      kvstar_topk                softmax-mass retrieval over block representatives
  kv_copy     Stream.Paged*Async         selected KV blocks out of the paged cache and back into fresh blocks

Codes in a cache are uniform random bits: what a random projection makes of centred keys.
"""
import math
import os
import sys

import numpy as np
import torch

# the package of the tree that is measured: the working folder is its root
sys.path.insert(0, os.path.join(os.getcwd(), "unified-cache-management_amd"))

from ucm_amd.sparse.decode_step import GSADecodeStep, GSADecodeStepMLA, SparseDecodeStep  # noqa: E402
from ucm_amd.sparse.esa_retrieval_worker import dot_topk  # noqa: E402
from ucm_amd.sparse.hash_encoder import HashEncoder  # noqa: E402
from ucm_amd.sparse.kvstar_retrieve import kvstar_topk  # noqa: E402
from ucm_amd.trans import Device  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
NOPE, ROPE = 512, 64  # the latent vector's and the rope part's dimensions; as many hash bits


def listed():
    return [
        # one chat at 8k tokens: a layer's decode step is all latency
        dict(name="gqa_decode_one", kind="gqa_decode", batch=1, context=8192, ragged=False, hq=32, hkv=8, dim=128,
             block=128, keep=2048, dtype="bf16"),
        # a full decode batch at 32k tokens
        dict(name="gqa_decode_batch", kind="gqa_decode", batch=32, context=32768, ragged=False, hq=32, hkv=8, dim=128,
             block=128, keep=8192, dtype="bf16"),
        # few long requests of very different lengths, a list and scores per KV head
        dict(name="gqa_topk_ragged", kind="gqa_topk", batch=8, context=131072, ragged=True, hq=32, hkv=8, dim=128,
             block=128, keep=16384, dtype="bf16"),
        # two requests of a latent-attention model, half precision
        dict(name="mla_decode_two", kind="mla_decode", batch=2, context=20000, ragged=True, hq=128, reduce=2, block=64,
             keep=2048, dtype="fp16"),
        # a decode batch of a latent-attention model at 64k tokens
        dict(name="mla_decode_batch", kind="mla_decode", batch=16, context=65536, ragged=False, hq=128, reduce=2,
             block=64, keep=8192, dtype="bf16"),
        # a prefill chunk as a serving engine schedules it
        dict(name="gqa_encode_chunk", kind="gqa_encode", tokens=2048, heads=8, dim=128, block=128, dtype="bf16"),
        # the cache of a 128k-token context built in one call
        dict(name="gqa_encode_build", kind="gqa_encode", tokens=131072, heads=8, dim=128, block=128, dtype="bf16"),
        # a prefill chunk of a latent-attention model
        dict(name="mla_encode_chunk", kind="mla_encode", tokens=8192, block=64, dtype="bf16"),
        # a 32k-token prefix found in the store, its last block part full
        dict(name="rehash_prefix", kind="rehash", tokens=32691, heads=8, dim=128, block=128, dtype="bf16"),
        # block vectors of a long document, two queries over 8000 candidates each
        dict(name="esa_two", kind="esa", batch=2, items=25600, dim=1024, candidates=8000, topk=3000),
        # 32k tokens as 64 merged representatives per block, a quarter of the channels, eight query tokens
        dict(name="kvstar_32k", kind="kvstar", tokens=8, hq=32, hkv=8, dim=128, kept=32, blocks=253, repre=64, topk=64),
        # 64 selected blocks of 32 layers' keys and values: out, and back into other blocks
        dict(name="kv_copy_blocks", kind="kv_copy", blocks=64, columns=64, column_bytes=262144),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gqa_decode", "gqa_topk", "mla_decode", "gqa_encode", "mla_encode", "rehash", "esa", "kvstar",
                       "kv_copy"])
    c = dict(kind=kind)
    if kind in ("gqa_decode", "gqa_topk"):
        c["batch"] = _log(rng, 1, 64)
        c["context"] = _log(rng, 4096, min(131072, 2 ** 21 // c["batch"]))
        c["ragged"] = rng.random() < 0.7
        c["hq"], c["hkv"] = rng.choice([(32, 8), (32, 8), (64, 8), (16, 4), (8, 8), (16, 2), (8, 1)])
        c["dim"] = rng.choice([128, 128, 64])
        c["block"] = rng.choice([128, 128, 64, 32])
        if c["block"] == 32:
            c["context"] = min(c["context"], 65536)
        c["keep"] = c["block"] * max(8, c["context"] // c["block"] // rng.choice([4, 8, 16]))
        c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
    elif kind == "mla_decode":
        c["batch"] = _log(rng, 1, 32)
        c["context"] = _log(rng, 4096, min(131072, 2 ** 21 // c["batch"]))
        c["ragged"] = rng.random() < 0.7
        c["hq"], c["reduce"] = rng.choice([(128, 2), (128, 1), (64, 1), (64, 2), (16, 2), (16, 1)])
        c["block"] = rng.choice([64, 64, 128])
        c["keep"] = c["block"] * max(8, c["context"] // c["block"] // rng.choice([4, 8, 16]))
        c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
    elif kind in ("gqa_encode", "rehash"):
        c["heads"] = rng.choice([8, 8, 4, 2, 1])
        c["tokens"] = _log(rng, 64, 2 ** 20 // c["heads"])
        c["dim"] = rng.choice([128, 128, 64])
        c["block"] = rng.choice([128, 128, 64, 32])
        c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        if c["dtype"] == "fp32":
            c["tokens"] = min(c["tokens"], 32768)
    elif kind == "mla_encode":
        c.update(tokens=_log(rng, 64, 131072), block=rng.choice([64, 64, 128]), dtype=rng.choice(["bf16", "bf16", "fp16"]))
    elif kind == "esa":
        c["batch"] = _log(rng, 1, 8)
        c["dim"] = rng.choice([128, 512, 1024, 1024, 1000])
        c["items"] = _log(rng, 1000, 60000)
        c["candidates"] = _log(rng, min(200, c["items"]), min(16000, c["items"]))
        c["topk"] = max(1, min(4096, int(c["candidates"] * rng.uniform(0.1, 0.5))))
    elif kind == "kvstar":
        c["tokens"] = rng.choice([1, 4, 8, 8, 16])
        c["hq"], c["hkv"] = rng.choice([(32, 8), (32, 8), (28, 4), (16, 2), (8, 8)])
        c["dim"] = 128
        c["kept"] = rng.choice([32, 32, 64, 128])
        c["blocks"] = _log(rng, 24, 1024)
        c["repre"] = rng.choice([64, 32, 16, 1])
        c["topk"] = max(4, c["blocks"] // rng.choice([3, 4, 8]))
    else:
        c["columns"] = rng.choice([2, 32, 56, 64])
        c["column_bytes"] = rng.choice([262144, 131072, 73728, 32768, 4096])
        c["blocks"] = _log(rng, 4, min(512, 2 ** 30 // (c["columns"] * c["column_bytes"])))
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _codes(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31, shape, dtype=torch.int32, device="cuda", generator=g)


def _normal(g, dtype, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _projection(g, dtype, *shape):
    return _normal(g, torch.float32, *shape).to(dtype)


def _lengths(case):
    """Token counts of the requests: all `context`, or spread from an eighth of it up to it.  A function of the
    case alone, so that every seed has the same work."""
    b, c = case["batch"], case["context"]
    if not case["ragged"]:
        return [c] * b
    return [c if i == 0 else c // 8 + (i * 2654435761 + 97) % (c - c // 8 + 1) for i in range(b)]


def _paged(g, case):
    """Block table, lengths, the slot of every request's last token, and the number of blocks."""
    bs = case["block"]
    lens = _lengths(case)
    need = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(need), generator=g, device="cuda").to(torch.int32)
    table = torch.zeros((len(lens), max(need)), dtype=torch.int32, device="cuda")
    first = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[first:first + n]
        first += n
    last = torch.tensor([(n - 1) // bs for n in lens], device="cuda")
    off = torch.tensor([(n - 1) % bs for n in lens], device="cuda")
    slots = table.gather(1, last[:, None])[:, 0].long() * bs + off
    return table, torch.tensor(lens, dtype=torch.int32, device="cuda"), slots, sum(need)


def _slots(g, tokens, block):
    """Slots of `tokens` consecutive tokens in blocks handed out in any order."""
    n = -(-tokens // block)
    ids = torch.randperm(n, generator=g, device="cuda")
    t = torch.arange(tokens, device="cuda")
    return ids[t // block] * block + t % block, ids.to(torch.int32), n


def _encoder(g, din, bits, dtype):
    enc = HashEncoder(din, bits, dtype, torch.device("cuda:0"))
    enc.set_hash_weight(_projection(g, dtype, din, bits))
    return enc


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("gqa_decode", "gqa_topk"):
        dt, d, hq, hkv = _DTYPES[case["dtype"]], case["dim"], case["hq"], case["hkv"]
        table, lens, slots, nb = _paged(g, case)
        b = case["batch"]
        cache = _codes(g, nb, case["block"], hkv, d // 32)
        keys, queries = _normal(g, dt, b, hkv, d), _normal(g, dt, b, hq, d)
        if kind == "gqa_decode":  # one projection for all heads, as the plugin has it
            step = GSADecodeStep(_projection(g, dt, d, d), hq, hkv, b, table.shape[1], case["keep"],
                                 block_size=case["block"])
        else:  # one projection per KV head
            step = SparseDecodeStep(_projection(g, dt, hkv, d, d), hq, hkv, b, table.shape[1],
                                    case["keep"] // case["block"], block_size=case["block"])
        return dict(kind=kind, step=step, args=(keys, slots, queries, cache, table, lens))
    if kind == "mla_decode":
        dt, hq, b = _DTYPES[case["dtype"]], case["hq"], case["batch"]
        table, lens, slots, nb = _paged(g, case)
        cache = _codes(g, nb, case["block"], (NOPE + ROPE) // 32)
        step = GSADecodeStepMLA(_projection(g, dt, NOPE, NOPE), _projection(g, dt, ROPE, ROPE), hq, case["reduce"], b,
                                table.shape[1], case["keep"], block_size=case["block"])
        args = (_normal(g, dt, b, NOPE), _normal(g, dt, b, ROPE), slots, _normal(g, dt, b, hq, NOPE),
                _normal(g, dt, b, hq, ROPE), cache, table, lens)
        return dict(kind=kind, step=step, args=args)
    if kind == "gqa_encode":
        dt, h, d = _DTYPES[case["dtype"]], case["heads"], case["dim"]
        slots, _, nb = _slots(g, case["tokens"], case["block"])
        cache = torch.zeros((nb, case["block"], h, d // 32), dtype=torch.int32, device="cuda")
        return dict(kind=kind, enc=_encoder(g, d, d, dt), keys=_normal(g, dt, case["tokens"], h, d), slots=slots,
                    cache=cache, block=case["block"])
    if kind == "mla_encode":
        dt, t = _DTYPES[case["dtype"]], case["tokens"]
        slots, _, nb = _slots(g, t, case["block"])
        cache = torch.zeros((nb, case["block"], 1, (NOPE + ROPE) // 8), dtype=torch.uint8, device="cuda")
        return dict(kind=kind, nope=_encoder(g, NOPE, NOPE, dt), rope=_encoder(g, ROPE, ROPE, dt),
                    k_nope=_normal(g, dt, t, 1, NOPE), k_rope=_normal(g, dt, t, 1, ROPE), slots=slots, cache=cache,
                    block=case["block"])
    if kind == "rehash":
        dt, h, d, bs = _DTYPES[case["dtype"]], case["heads"], case["dim"], case["block"]
        _, ids, nb = _slots(g, case["tokens"], bs)
        return dict(kind=kind, enc=_encoder(g, d, d, dt), kv=_normal(g, dt, nb, bs, h, d), ids=ids,
                    tokens=case["tokens"], cache=torch.zeros((nb, bs, h, d // 32), dtype=torch.int32, device="cuda"),
                    block=bs)
    if kind == "esa":
        n, d, b = case["items"], case["dim"], case["batch"]
        idx = torch.stack([torch.randperm(n, generator=g, device="cuda")[:case["candidates"]] for _ in range(b)])
        return dict(kind=kind, data=_normal(g, torch.float32, n, d), query=_normal(g, torch.float32, b, d),
                    idx=idx.to(torch.int32), topk=case["topk"])
    if kind == "kvstar":
        q = _normal(g, torch.float16, case["tokens"], case["hq"], case["dim"]) * 0.5
        k = _normal(g, torch.float16, case["blocks"], case["repre"], case["hkv"], case["kept"]) * 0.5
        pruned = None
        if case["kept"] < case["dim"]:
            order = torch.rand(case["hkv"], case["dim"], generator=g, device="cuda").argsort(dim=1)
            pruned = order[:, :case["kept"]].sort(dim=1).values.contiguous()
        return dict(kind=kind, q=q, k=k, pruned=pruned, topk=case["topk"])
    # kv_copy: keys / values of every layer are columns of one paged cache; the blocks come back elsewhere
    n, cols, cb = case["blocks"], case["columns"], case["column_bytes"]
    nb = 2 * n + 3
    kv = torch.empty((cols, nb, cb // 2), dtype=torch.int16, device="cuda").random_(generator=g)
    ids = torch.randperm(nb, generator=g, device="cuda").to(torch.int32).cpu().numpy()
    dev = Device()
    dev.Setup(0)
    base = np.array([kv[c].data_ptr() for c in range(cols)], np.uint64)
    return dict(kind=kind, kv=kv, flat=torch.empty((n, cols, cb // 2), dtype=torch.int16, device="cuda"),
                stream=dev.MakeSMStream(), base=base, sizes=np.full(cols, cb, np.uint64), taken=ids[:n],
                fresh=ids[n:2 * n], nb=nb)


def run(s):
    kind = s["kind"]
    if kind in ("gqa_decode", "gqa_topk"):
        return (*s["step"].step(*s["args"]), s["args"][3])
    if kind == "mla_decode":
        return (*s["step"].step(*s["args"]), s["args"][5])
    if kind == "gqa_encode":
        return s["enc"].compute_hash_and_cache(s["keys"], s["slots"], s["cache"], block_size=s["block"])
    if kind == "mla_encode":
        s["nope"].compute_hash_and_cache(s["k_nope"], s["slots"], s["cache"][..., :NOPE // 8], block_size=s["block"])
        s["rope"].compute_hash_and_cache(s["k_rope"], s["slots"], s["cache"][..., NOPE // 8:], block_size=s["block"])
        return s["cache"]
    if kind == "rehash":
        return s["enc"].compute_hash_from_paged_cache(s["kv"], s["ids"], s["tokens"], s["cache"], block_size=s["block"])
    if kind == "esa":
        return dot_topk(s["data"], s["query"], s["idx"], s["topk"])
    if kind == "kvstar":
        return kvstar_topk(s["q"], s["k"], s["pruned"], s["topk"])
    st = s["stream"]
    st.PagedGatherAsync(s["base"], s["sizes"], s["taken"], s["flat"].data_ptr(), num_cache_blocks=s["nb"])
    st.PagedScatterAsync(s["flat"].data_ptr(), s["base"], s["sizes"], s["fresh"], sync=True, num_cache_blocks=s["nb"])
    return s["flat"], s["kv"]


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype") == "fp32" else 2
    if kind in ("gqa_decode", "gqa_topk"):
        b, d, hq, hkv = case["batch"], case["dim"], case["hq"], case["hkv"]
        lens = _lengths(case)
        blocks = sum(-(-n // case["block"]) for n in lens)
        rows = b * hkv + b * (hq if kind == "gqa_topk" else hkv)  # projections: new keys, and queries or their means
        w = d * d * (hkv if kind == "gqa_topk" else 1) * size
        out = b * (max(lens) // case["block"] + 1) * 4 if kind == "gqa_decode" else b * hkv * case["keep"] // case["block"] * 8
        return {"bytes": sum(lens) * hkv * d / 8 + 4 * blocks + b * (hkv + hq) * d * size + w + b * hkv * d / 8 + out,
                "flops": 2.0 * rows * d * d}
    if kind == "mla_decode":
        b, hq = case["batch"], case["hq"]
        lens = _lengths(case)
        blocks = sum(-(-n // case["block"]) for n in lens)
        rows = b + b * hq // case["reduce"]
        return {"bytes": sum(lens) * 72 + 4 * blocks + b * (1 + hq) * (NOPE + ROPE) * 2 + (NOPE ** 2 + ROPE ** 2) * 2
                + 4 * b * (max(lens) // case["block"] + 1), "flops": 2.0 * rows * (NOPE ** 2 + ROPE ** 2)}
    if kind in ("gqa_encode", "rehash"):
        rows, d = case["tokens"] * case["heads"], case["dim"]
        index = case["tokens"] * 8 if kind == "gqa_encode" else case["tokens"] // case["block"] * 4
        return {"bytes": rows * (d * size + d / 8) + index + d * d * size, "flops": 2.0 * rows * d * d}
    if kind == "mla_encode":
        t = case["tokens"]
        return {"bytes": t * ((NOPE + ROPE) * 2 + 72 + 8) + (NOPE ** 2 + ROPE ** 2) * 2,
                "flops": 2.0 * t * (NOPE ** 2 + ROPE ** 2)}
    if kind == "esa":
        pairs = case["batch"] * case["candidates"]
        rows = min(pairs, case["items"])
        return {"bytes": rows * case["dim"] * 4.0 + 4 * pairs + 8 * case["batch"] * case["topk"], "flops": 2.0 * pairs * case["dim"]}
    if kind == "kvstar":
        reps, rows = case["blocks"] * case["repre"], case["tokens"] * case["hq"]
        return {"bytes": reps * case["hkv"] * case["kept"] * 2.0 + rows * case["dim"] * 2 + 8 * case["topk"],
                "flops": 2.0 * rows * reps * case["kept"]}
    return {"bytes": 4.0 * case["blocks"] * case["columns"] * case["column_bytes"], "flops": 0.0}


def tolerance(case):
    """Compared with the same paths in 64 bits: code words differ only where a projection is within rounding of zero
    (at most 2.4e-6 of them: four times that, and one word of a small output); float sums in another order move scores
    by 1.1e-7 of their norm and 4e-7 of their mean size, which changes places of neighbours (0.15 % seen)."""
    kind = case["kind"]
    if kind in ("gqa_encode", "rehash"):
        return {"rel": 0.0, "differ": 1e-5 + 32.0 / (case["tokens"] * case["heads"] * case["dim"])}
    if kind == "mla_encode":
        return {"rel": 0.0, "differ": 1e-5 + 1.0 / (case["tokens"] * 72)}
    if kind in ("esa", "kvstar"):
        return {"rel": 5e-7, "max": 2e-6, "differ": 6e-3}
    return "exact"  # integer scores of codes whose projections keep clear of zero
