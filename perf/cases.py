"""Timed work of the split decode path: what a serving program has it do, layer by layer.

Every case is one call (or one layer's calls) of the package's public entry
points on inputs already on the GPU:

  decode   ops.paged_decode over the HBM tier in vLLM's interleaved layout:
           the attention of one layer for one decode step. Rows' lengths are
           uniform in [lo, hi] tokens, their blocks scattered over the pool.
           "planned" rows come with what the step's planner knows on the host
           (the dispatch order, the token total); the others with the tables
           and lengths alone, as flash_attn_varlen_func's caller gives them.
           "capacity" > 0: the block table is as wide as the longest context
           the server admits, and the call says how long the longest row is.
  layer    SplitDecodeImpl._forward_device: one layer of a step planned on the
           GPU, with some of the rows' newest blocks in the pinned host tier:
           both tiers' cache writes, the fused two-tier decode, the output rows.
  hybrid   ops.hybrid_split_decode: a decode step whose host tier is large, its
           blocks shared between the host cores and the GPU.
  write    ops.reshape_and_cache: the KV rows of a prefill (or of a decode
           step) into the HBM tier.

Lengths depend on the case alone (so its work is known without its inputs);
the seed decides which row has which length, where the blocks lie, and the
values, N(0, 1) as in the repository's workloads.
"""

from __future__ import annotations

import math
import random

import torch

from vllm_fastdecoder_amd import backend, ops, state
from vllm_fastdecoder_amd.pinned import pinned_empty

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
BLOCK_SIZES = (16, 32, 64)
# (query heads, kv heads, head size) of the decode cases: multi-head, grouped
# and tensor-parallel shares of them, at the head sizes in common use
LAYOUTS = ((32, 32, 128), (32, 8, 128), (28, 4, 128), (8, 1, 128), (16, 8, 256), (32, 32, 80),
           (32, 32, 64), (14, 2, 64), (16, 2, 96), (40, 8, 128))
LARGEST_BYTES = 2_650_000_000  # the Llama-3-8B decode below


def _decode(name, n, heads, dtype, lo, hi, bs=16, planned=True, capacity=0):
    H, KVH, D = heads
    return {"name": name, "kind": "decode", "n": n, "H": H, "KVH": KVH, "D": D, "BS": bs,
            "dtype": dtype, "lo": lo, "hi": hi, "planned": planned, "capacity": capacity}


def listed() -> list[dict]:
    return [
        # one interactive user: the smallest call, where latency counts
        _decode("decode_one_user", 1, (32, 8, 128), "bf16", 900, 900, planned=False, capacity=8192),
        # a handful of users with short contexts (the repository's small batch)
        _decode("decode_small_batch", 8, (32, 32, 128), "fp16", 128, 1024),
        # a full batch of a multi-head model (the repository's vicuna-7b workload)
        _decode("decode_mha_full_batch", 128, (32, 32, 128), "fp16", 256, 2048),
        # a full batch of a grouped-query model (the repository's Llama-3-8B workload)
        _decode("decode_gqa_full_batch", 256, (32, 8, 128), "bf16", 1024, 4096),
        # a few very long documents of uneven length
        _decode("decode_long_documents", 3, (32, 8, 128), "bf16", 12_000, 50_000, planned=False),
        # one GPU's share of a large grouped-query model under 8-way tensor parallelism
        _decode("decode_tensor_parallel", 64, (8, 1, 128), "bf16", 1024, 4096),
        # a mid-sized batch of a grouped-query model, contexts from new to long,
        # 32-token blocks, the table at the server's capacity
        _decode("decode_mixed_lengths", 40, (28, 4, 128), "bf16", 50, 3100, bs=32, capacity=8192),
        # head size 256, two query heads per kv head
        _decode("decode_head_256", 24, (16, 8, 256), "bf16", 200, 4000, planned=False),
        # fp32 caches, the reference's third data type
        _decode("decode_fp32", 12, (32, 8, 128), "fp32", 64, 1500),
        # one layer of a step whose newest tokens spilled to the host tier
        {"name": "layer_two_tiers", "kind": "layer", "n": 33, "H": 32, "KVH": 8, "D": 128,
         "BS": 16, "dtype": "bf16", "lo": 40, "hi": 1800, "host_blocks": 1},
        # a step with most of its KV in host memory: host cores and GPU together
        {"name": "hybrid_host_heavy", "kind": "hybrid", "n": 24, "H": 32, "KVH": 32, "D": 128,
         "BS": 16, "dtype": "fp16", "lo": 256, "hi": 1024, "share": 0.875},
        # a prefill chunk's KV rows (vLLM's slot mapping: padding rows are -1)
        {"name": "write_prefill", "kind": "write", "T": 8101, "KVH": 8, "D": 128, "BS": 16,
         "dtype": "bf16"},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    """Another case of the same ranges: mostly decode calls, sizes spread over
    their logarithm."""
    pick = rng.random()
    if pick < 0.08:
        return {"kind": "write", "T": _log_int(rng, 1, 16_384), "KVH": rng.choice((1, 4, 8, 32)),
                "D": rng.choice((64, 80, 128, 256)), "BS": rng.choice(BLOCK_SIZES),
                "dtype": rng.choice(("fp16", "bf16"))}
    if pick < 0.2:
        lo = _log_int(rng, 32, 1000)
        return {"kind": "layer", "n": _log_int(rng, 1, 96), "H": 32, "KVH": rng.choice((8, 32)),
                "D": 128, "BS": rng.choice((16, 32)), "dtype": rng.choice(("fp16", "bf16")),
                "lo": lo, "hi": 2 * lo + rng.randrange(32), "host_blocks": 1}
    while True:
        H, KVH, D = rng.choice(LAYOUTS)
        lo = _log_int(rng, 16, 16_000)
        hi = lo + int(lo * rng.choice((0.0, 0.5, 1.0, 3.0, 7.0))) + rng.randrange(16)
        dtype = rng.choice(("fp16", "bf16", "bf16", "fp32"))
        case = {"kind": "decode", "n": _log_int(rng, 1, 256), "H": H, "KVH": KVH, "D": D,
                "BS": rng.choice(BLOCK_SIZES), "dtype": dtype, "lo": lo, "hi": hi,
                "planned": rng.random() < 0.6,
                "capacity": rng.choice((0, 0, max(8192, 2 * hi)))}
        if work(case)["bytes"] <= LARGEST_BYTES:
            return case


# ------------------------------------------------------------------ inputs


def _elt(case) -> int:
    return DTYPES[case["dtype"]].itemsize


def _lens(case) -> list[int]:
    """The rows' lengths, a function of the case alone: an even spread of [lo, hi] with jitter."""
    n, lo, hi = case["n"], case["lo"], case["hi"]
    rng = random.Random(97 * n + 31 * lo + hi)
    return [rng.randint(lo, hi) for _ in range(n)]


def _blocks(tokens: int, bs: int) -> int:
    return -(-tokens // bs)


class _Draws:
    """Seeded values: small things on the CPU, caches straight on the GPU."""

    def __init__(self, seed: int):
        self.cpu = torch.Generator().manual_seed(seed)
        self.gpu = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, dtype) -> torch.Tensor:
        out = torch.empty(shape, dtype=dtype, device="cuda")
        rows = max(1, (1 << 28) // max(1, out[0].numel()))
        for s in range(0, shape[0], rows):  # in slabs: the fp32 draw stays small
            part = out[s:s + rows]
            part.copy_(torch.randn(part.shape, generator=self.gpu, device="cuda"))
        return out

    def order(self, items: list) -> list:
        return [items[i] for i in torch.randperm(len(items), generator=self.cpu).tolist()]

    def tables(self, counts: list[int], width: int, pool: int) -> torch.Tensor:
        """Each row's blocks: distinct ids scattered over the pool."""
        perm = torch.randperm(pool, generator=self.cpu).to(torch.int32)
        bt = torch.zeros(len(counts), max(width, 1), dtype=torch.int32)
        pos = 0
        for i, c in enumerate(counts):
            bt[i, :c] = perm[pos:pos + c]
            pos += c
        return bt


def _hbm_cache(draws, pool, case):
    kv = draws.normal((max(pool, 1), case["BS"], case["KVH"], 2 * case["D"]), DTYPES[case["dtype"]])
    return kv, kv[..., :case["D"]], kv[..., case["D"]:]


def _to_host_tier(draws, pool, case):
    """K and V of the pinned host tier [C, KVH, BS, D]."""
    shape = (max(pool, 1), case["KVH"], case["BS"], case["D"])
    pair = []
    for _ in range(2):
        t = pinned_empty(shape, DTYPES[case["dtype"]])
        t.copy_(draws.normal(shape, DTYPES[case["dtype"]]).cpu())
        pair.append(t)
    return pair


def prepare(case, seed):
    draws = _Draws(seed)
    return {"decode": _prepare_decode, "layer": _prepare_layer, "hybrid": _prepare_hybrid,
            "write": _prepare_write}[case["kind"]](case, draws)


def _prepare_decode(case, draws):
    bs = case["BS"]
    lens = draws.order(_lens(case))
    counts = [_blocks(x, bs) for x in lens]
    pool = sum(counts)
    width = _blocks(max(case["capacity"], max(lens)), bs)
    kv, kc, vc = _hbm_cache(draws, pool, case)
    st = {"case": case, "kv": kv, "k": kc, "v": vc, "lens_list": lens,
          "bt": draws.tables(counts, width, pool).cuda(),
          "lens": torch.tensor(lens, dtype=torch.int32).cuda(),
          "q": draws.normal((case["n"], case["H"], case["D"]), DTYPES[case["dtype"]]),
          "max": max(lens), "order": None, "total": None}
    if case["planned"]:
        st["order"] = ops.longest_first(torch.tensor(lens, dtype=torch.int32)).cuda()
        st["total"] = sum(lens)
    return st


def _prepare_layer(case, draws):
    """A decode step of n rows, each row's newest `host_blocks` blocks (with
    the token being decoded) in the host tier, the rest in HBM."""
    n, bs, KVH, D = case["n"], case["BS"], case["KVH"], case["D"]
    dt = DTYPES[case["dtype"]]
    lens = draws.order(_lens(case))
    counts = [_blocks(x, bs) for x in lens]
    host = [min(case["host_blocks"], c) for c in counts]
    hbm = [c - h for c, h in zip(counts, host)]
    G, C = max(sum(hbm), 1), max(sum(host), 1)
    t_hbm = draws.tables(hbm, max(counts), G)
    t_host = draws.tables(host, case["host_blocks"], C)
    bt = torch.zeros(n, max(counts), dtype=torch.int32)
    slots = []
    for i in range(n):
        bt[i, :hbm[i]] = t_hbm[i, :hbm[i]]
        bt[i, hbm[i]:counts[i]] = t_host[i, :host[i]] + G
        slots.append(int(bt[i, counts[i] - 1]) * bs + (lens[i] - 1) % bs)
    kv, _, _ = _hbm_cache(draws, G, case)
    hk, hv = _to_host_tier(draws, C, case)
    store = state.HostKVStore(G, C, bs, KVH, D, dt, k={"layer": hk}, v={"layer": hv})
    step = backend.build_device_step(
        torch.arange(n + 1, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32), bt.cuda(),
        torch.tensor(slots, dtype=torch.int64).cuda(), n, store, torch.device("cuda"))
    layer = type("Layer", (), {"layer_name": "layer"})()
    impl = backend.SplitDecodeImpl(case["H"], KVH, D, 1.0 / math.sqrt(D))
    q = draws.normal((n, case["H"], D), dt)
    k, v = draws.normal((n, KVH, D), dt), draws.normal((n, KVH, D), dt)
    return {"case": case, "store": store, "kv": kv, "kv_view": kv.permute(0, 2, 1, 3), "hk": hk,
            "hv": hv, "step": step, "layer": layer, "impl": impl, "q": q, "key": k, "value": v,
            "out": torch.empty_like(q), "lens_list": lens, "counts": counts, "bt": bt, "G": G,
            "slots": slots}


def _prepare_hybrid(case, draws):
    """The last 60 % of each row's blocks in the pinned host tier."""
    bs = case["BS"]
    lens = draws.order(_lens(case))
    counts = [_blocks(x, bs) for x in lens]
    host = [math.ceil(0.6 * c) for c in counts]
    hbm = [c - h for c, h in zip(counts, host)]
    G, C = max(sum(hbm), 1), max(sum(host), 1)
    kv, kc, vc = _hbm_cache(draws, G, case)
    hk, hv = _to_host_tier(draws, C, case)
    return {"case": case, "kv": kv, "k": kc, "v": vc, "hk": hk, "hv": hv, "lens_list": lens,
            "bt_hbm": draws.tables(hbm, max(hbm), G), "bt_host": draws.tables(host, max(host), C),
            "lens_hbm": torch.tensor([h * bs for h in hbm], dtype=torch.int32),
            "lens_host": torch.tensor([x - h * bs for x, h in zip(lens, hbm)], dtype=torch.int32),
            "q": draws.normal((case["n"], case["H"], case["D"]), DTYPES[case["dtype"]])}


def _prepare_write(case, draws):
    """T tokens into scattered blocks (consecutive slots inside a block), every
    64th a padding row."""
    T, bs = case["T"], case["BS"]
    nb = _blocks(T, bs)
    kv, kc, vc = _hbm_cache(draws, nb + 3, case)
    ids = draws.tables([nb], nb, nb + 3)[0].to(torch.int64)
    tok = torch.arange(T)
    slots = ids[tok // bs] * bs + tok % bs
    slots[63::64] = -1
    dt = DTYPES[case["dtype"]]
    return {"case": case, "kv": kv, "k": kc, "v": vc, "slots": slots.cuda(),
            "key": draws.normal((T, case["KVH"], case["D"]), dt),
            "value": draws.normal((T, case["KVH"], case["D"]), dt)}


# ------------------------------------------------------------------ one pass


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        return ops.paged_decode(st["q"], st["k"], st["v"], st["bt"], st["lens"],
                                1.0 / math.sqrt(case["D"]), row_order=st["order"],
                                max_seqlen_k=st["max"], total_tokens=st["total"])
    if kind == "layer":
        state.STORE = st["store"]  # the worker's store: one per process
        out = st["impl"]._forward_device(st["layer"], st["q"], st["key"], st["value"],
                                         st["kv_view"], st["step"], st["out"])
        return out, st["kv"], st["hk"], st["hv"]
    if kind == "hybrid":
        return ops.hybrid_split_decode(st["q"], st["k"], st["v"], st["bt_hbm"], st["lens_hbm"],
                                       st["hk"], st["hv"], st["bt_host"], st["lens_host"],
                                       1.0 / math.sqrt(case["D"]), case["share"])
    ops.reshape_and_cache(st["key"], st["value"], st["k"], st["v"], st["slots"])
    return st["kv"]


def work(case):
    """K and V of every row's tokens, q, out, lse, the ids and lengths, each
    once; a layer also its new KV rows (read and written)."""
    elt = _elt(case)
    if case["kind"] == "write":
        rows = case["T"] - case["T"] // 64
        return {"bytes": 4 * rows * case["KVH"] * case["D"] * elt + 8 * case["T"], "flops": 0}
    lens = _lens(case)
    n, H, KVH, D = case["n"], case["H"], case["KVH"], case["D"]
    tokens = sum(lens)
    nbytes = (2 * tokens * KVH * D * elt + 2 * n * H * D * elt + 4 * n * H + 4 * n
              + 4 * sum(_blocks(x, case["BS"]) for x in lens))
    if case["kind"] == "layer":
        nbytes += 4 * n * KVH * D * elt - 4 * n * H + 8 * n
    return {"bytes": nbytes, "flops": 4 * tokens * H * D}


def tolerance(case):
    """Four times the distance from 64 bits seen: 1.7e-3 bf16 and 2.1e-4 fp16
    (the outputs' last rounding), 1.8e-7 fp32 at up to 1,500 tokens a row, with
    room for the sums of rows of 100,000. Bytes that are only moved stay the same."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": {"bf16": 7e-3, "fp16": 1e-3, "fp32": 2e-6}[case["dtype"]]}


# ------------------------------------------------------------------ in 64 bits


def _attend(q, k, v, scale):
    """q [H, D], k and v [L, KVH, D] in float64 -> out [H, D], lse [H]."""
    H, D = q.shape
    KVH = k.shape[1]
    kk = k.permute(1, 2, 0).contiguous()
    vv = v.permute(1, 0, 2).contiguous()
    s = torch.matmul(q.reshape(KVH, H // KVH, D) * scale, kk)
    lse = torch.logsumexp(s, dim=-1)
    p = torch.exp(s - lse[..., None])
    return torch.matmul(p, vv).reshape(H, D), lse.reshape(H)


def _rows(cache, table, count, length):
    """A row's tokens [length, KVH, D] of a [B, BS, KVH, D] view, in float64."""
    got = cache[table[:count].to(cache.device).long()].to("cuda").double()
    return got.flatten(0, 1)[:length]


def exact(case, seed):
    if case["kind"] == "write":
        return None
    st = prepare(case, seed)
    n, D, bs = case["n"], case["D"], case["BS"]
    scale = 1.0 / math.sqrt(D)
    outs, lses = [], []
    if case["kind"] == "layer":  # the step's tokens are written before they are read
        kc, vc = st["kv"][..., :D], st["kv"][..., D:]
        hk, hv = st["hk"].transpose(1, 2), st["hv"].transpose(1, 2)
        for i, slot in enumerate(st["slots"]):
            b, off = slot // bs, slot % bs
            for hbm, host, row in ((kc, hk, st["key"]), (vc, hv, st["value"])):
                if b < st["G"]:
                    hbm[b, off] = row[i]
                else:
                    host[b - st["G"], off] = row[i].cpu()
    for i in range(n):
        L, q = st["lens_list"][i], st["q"][i].double()
        if case["kind"] == "decode":
            bt = st["bt"][i]
            k = _rows(st["k"], bt, _blocks(L, bs), L)
            v = _rows(st["v"], bt, _blocks(L, bs), L)
        elif case["kind"] == "layer":
            ids = st["bt"][i, :st["counts"][i]]
            a, b = ids[ids < st["G"]], ids[ids >= st["G"]] - st["G"]
            k, v = (torch.cat([_rows(x, a, len(a), len(a) * bs), _rows(y, b, len(b), len(b) * bs)])[:L]
                    for x, y in ((kc, hk), (vc, hv)))
        else:
            la, lb = int(st["lens_hbm"][i]), int(st["lens_host"][i])
            k, v = (torch.cat([_rows(x, st["bt_hbm"][i], _blocks(la, bs), la),
                               _rows(y.transpose(1, 2), st["bt_host"][i], _blocks(lb, bs), lb)])
                    for x, y in ((st["k"], st["hk"]), (st["v"], st["hv"])))
        o, l = _attend(q, k, v, scale)
        outs.append(o)
        lses.append(l)
    out = torch.stack(outs)
    if case["kind"] == "layer":
        return out, None, None, None
    return out, torch.stack(lses, dim=1)
