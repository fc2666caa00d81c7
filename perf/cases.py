"""What the KV data path is timed on: the work a serving program has it do, as plain cases.

A case names one of five kinds of work and its sizes:

  append   one model step's new keys / values written into the paged cache, one call per layer as a forward makes
           them (``cache_ops.reshape_and_cache_flash`` / ``cache_ops.reshape_and_cache``); ``tables``: the step
           starts from the block tables (``cache_ops.compute_slot_mapping``) instead of a finished slot mapping
  handoff  requests handed from one instance's pool to another's through transfer buffers: every request packed
           (``KVWorker.extract_kv_blocks``), then every buffer unpacked (``KVWorker.write_kv_blocks``, or
           ``kv_ops.kv_unpack_dequant_fp8`` where an fp8 pool feeds a 16-bit one)
  move     the same hand-over inside one device without buffers (``KVTransferManager``, CUDA_IPC)
  copy     blocks copied inside one pool (``cache_ops.copy_blocks``), as rescheduling does
  gather   cached vision embeddings of a batch concatenated (``KVWorker.gather_vision_embeddings``)

Pools are one allocation with per-layer views (``KVWorker.init_kvcache``'s default). All results are bytes moved
or rounded by a fixed rule, so every tolerance is exact.
"""
import math

import torch

from elasticmm_amd import cache_ops, kv_ops
from elasticmm_amd.kv_transfer import KVTransferManager, TransferMethod
from elasticmm_amd.worker import KVWorker

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "u8": torch.uint8}


def _append(name, **kw):
    case = {"name": name, "kind": "append", "layout": "flash", "cache": "auto", "dtype": "bf16", "layers": 28, "heads": 4,
            "dim": 128, "block": 16, "seqs": 0, "chunk": 0, "prompt": 0, "pad": 0.0, "slots": "prompts", "qkv": False,
            "tables": False, "blocks": 4000}
    case.update(kw)
    return case


def _handoff(name, **kw):
    case = {"name": name, "kind": "handoff", "dtype": "bf16", "layers": 28, "heads": 4, "dim": 128, "block": 16,
            "requests": 1, "least": 15, "most": 15, "tables": "list", "dequant": False, "blocks": 4000}
    case.update(kw)
    return case


def listed():
    return [
        # The smallest step: two dozen running sequences decode one token each. The step starts from their block
        # tables; K and V are views of the fused QKV projection's output (28 + 4 + 4 heads), as a forward has them.
        _append("decode_from_tables", seqs=24, qkv=True, tables=True),
        # Chunked prefill with decode tokens beside it: 256 sequences x 1 token and one chunk of 8192, slots random
        # over the free slots, 5 % of the entries padded with -1.
        _append("step_flash", seqs=256, chunk=8192, pad=0.05, slots="random"),
        # A full decode batch into the transposed paged-attention layout: every token alone in its block.
        _append("decode_paged", layout="paged", seqs=256, qkv=True),
        # Chunked prefill + decode in that layout: prompts fill blocks in order, decode tokens do not.
        _append("step_paged", layout="paged", seqs=256, chunk=8192, prompt=1536),
        # The quantising append of a 70B-class per-GPU shape (80 layers, 8 KV heads, fp8 cache).
        _append("step_fp8", cache="fp8", layers=80, heads=8, seqs=256, chunk=8192, prompt=3000, blocks=2500),
        # The fp8 cache in the paged-attention layout, saturating as that layout's own writers do; a smaller step.
        _append("step_fp8_paged", layout="paged", cache="fp8_sat", layers=80, heads=8, seqs=128, chunk=2048, prompt=700,
                blocks=2500),
        # One short request handed over (15 blocks): the launches and the host work in front of them.
        _handoff("handoff_short"),
        # A migrating batch: 32 requests of 512-4096 prompt tokens, each with a 1024-token image prefix. The largest.
        _handoff("handoff_batch", requests=32, least=96, most=320, blocks=12000),
        # An fp8 instance feeds a bf16 one: fp8 bytes packed, dequantised while they are unpacked.
        _handoff("handoff_fp8_dequant", dtype="u8", layers=80, heads=8, requests=4, least=64, most=512, dequant=True, blocks=2500),
        # Requests moved between two instances on one device by the transfer manager, block tables as lists.
        {"name": "move_requests", "kind": "move", "dtype": "bf16", "layers": 28, "heads": 4, "dim": 128, "block": 16,
         "requests": 8, "least": 30, "most": 300, "blocks": 6000},
        # Elastic rebalancing inside one pool: half of the live blocks go to free ones.
        {"name": "rebalance", "kind": "copy", "dtype": "bf16", "layers": 28, "heads": 4, "dim": 128, "block": 16,
         "pairs": 4500, "blocks": 12000},
        # The vision embeddings of 128 cached images, 64-2304 patches each, into one prefill input.
        {"name": "vision_gather", "kind": "gather", "dtype": "bf16", "hidden": 3584, "images": 128, "least": 64, "most": 2304},
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["append", "append", "append", "append", "append", "handoff", "handoff", "handoff", "move", "copy", "gather"])
    if kind == "gather":
        return {"kind": "gather", "dtype": rng.choice(["bf16", "f16"]), "hidden": rng.choice([1024, 1280, 3584]),
                "images": _between(rng, 2, 128), "least": 64, "most": _between(rng, 128, 2304)}
    shape = {"layers": rng.choice([24, 28, 32, 48]), "heads": rng.choice([2, 4, 8]), "dim": rng.choice([64, 128]), "block": 16}
    if kind == "append":
        layout = rng.choice(["flash", "paged"])
        cache = rng.choice(["auto", "auto", "fp8", "fp8_sat"])
        seqs = _between(rng, 1, 512)
        chunk = _between(rng, 33, 8192) if rng.random() < 0.6 else 0
        c = _append("", layout=layout, cache=cache, dtype=rng.choice(["bf16", "bf16", "f16"]), seqs=seqs, chunk=chunk,
                    prompt=_between(rng, 33, 4096), pad=rng.choice([0.0, 0.05]), qkv=rng.random() < 0.5,
                    slots=rng.choice(["prompts", "prompts", "random"]) if layout == "flash" else "prompts")
        c.update(shape, tables=c["slots"] == "prompts" and rng.random() < 0.3)
        c["blocks"] = 3000
    elif kind == "handoff":
        dequant = rng.random() < 0.3
        most = _between(rng, 2, 320)
        c = _handoff("", dtype="u8" if dequant else rng.choice(["bf16", "f16", "u8"]), requests=_between(rng, 1, 16),
                     least=max(1, most // rng.choice([1, 2, 5])), most=most, tables=rng.choice(["list", "list", "device"]), dequant=dequant)
        c.update(shape)
        c["blocks"] = max(1000, 2 * c["requests"] * most)
        while c["layers"] * c["heads"] * c["dim"] * c["blocks"] > 28 * 4 * 128 * 12000:  # no larger than the listed ones
            c["requests"] = max(1, c["requests"] // 2)
            c["blocks"] = max(1000, 2 * c["requests"] * most)
            if c["requests"] == 1:
                break
    elif kind == "move":
        most = _between(rng, 2, 320)
        c = {"kind": "move", "dtype": rng.choice(["bf16", "f16"]), "requests": _between(rng, 1, 8), "least": max(1, most // 4), "most": most}
        c.update(shape)
        c["blocks"] = max(1000, 2 * c["requests"] * most)
    else:
        pairs = _between(rng, 3, 2500)
        c = {"kind": "copy", "dtype": rng.choice(["bf16", "f16"]), "pairs": pairs}
        c.update(shape)
        c["blocks"] = max(1000, int(2.5 * pairs))
    c.pop("name", None)
    return c


# ---- sizes that follow from a case alone -------------------------------------------------------------------------
def _spread(count, least, most, salt):
    """`count` whole numbers in [least, most], spread evenly but in no order (a fixed rule: work() needs them too)."""
    return [least + int((most - least + 1) * ((0.5 + salt + i * 0.6180339887498949) % 1.0)) for i in range(count)]


def _step_lengths(case):
    """Query lengths of the step: decode sequences, then the prompts the chunk is made of."""
    left, prompts = case["chunk"], []
    while left > 0:
        q = min(left, case["prompt"] or left)
        prompts.append(q)
        left -= q
    return [1] * case["seqs"] + prompts


def _row(case):
    return case["heads"] * case["dim"]


def _block_counts(case):
    return _spread(case["requests"], case["least"], case["most"], 0.1)


# ---- inputs ------------------------------------------------------------------------------------------------------
def _generators(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed), torch.Generator().manual_seed(seed)


def _filled(shape, dtype, g):
    t = torch.empty(shape, dtype=dtype, device=DEVICE)
    if dtype == torch.uint8:  # fp8-e4m3 bytes of N(0, 1) values
        flat = t.view(-1)
        for i in range(0, flat.numel(), 1 << 28):
            part = flat[i:i + (1 << 28)]
            part.copy_(torch.randn(part.numel(), dtype=torch.float16, device=DEVICE, generator=g).to(torch.float8_e4m3fn).view(torch.uint8))
        return t
    return t.normal_(0.0, 0.5, generator=g)


def _pool(case, dtype, g):
    """(whole pool, its per-layer views): [layers, 2, blocks, block, heads, dim]."""
    whole = _filled((case["layers"], 2, case["blocks"], case["block"], case["heads"], case["dim"]), dtype, g)
    return whole, list(whole.unbind(0))


def _worker(case, dtype, g, rank):
    whole, layers = _pool(case, dtype, g)
    w = KVWorker(rank, DEVICE, case["block"])
    w.bind_kv_cache(layers)
    return whole, w


def _prepare_append(case, g, host):
    L, H, D, bs, NB = case["layers"], case["heads"], case["dim"], case["block"], case["blocks"]
    dt = DTYPES[case["dtype"]]
    cache_dt = dt if case["cache"] == "auto" else torch.uint8
    lengths = _step_lengths(case)
    total = sum(lengths)
    tokens = total + int(round(case["pad"] * total))
    # block tables: disjoint random blocks per sequence; decode sequences sit somewhere inside their last block
    perm = torch.randperm(NB, generator=host).tolist()
    tables, contexts, at = [], [], 0
    for q in lengths:
        ctx = int(torch.randint(0, bs, (1,), generator=host)) if q == 1 else 0
        n = (ctx + q + bs - 1) // bs
        tables.append(perm[at:at + n])
        contexts.append(ctx)
        at += n
    if case["slots"] == "random":
        slots = torch.full((tokens,), -1, dtype=torch.long)
        where = torch.randperm(tokens, generator=host)[:total]
        slots[where] = torch.randperm(NB * bs, generator=host)[:total]
        slots = slots.to(DEVICE)
    else:
        slots = cache_ops.compute_slot_mapping(tables, contexts, lengths, bs, pad_to=tokens, device=torch.device(DEVICE))
    if case["qkv"]:  # views of the fused projection's output, 7 query heads per KV head
        wide = torch.empty((L, tokens, 9 * H * D), dtype=dt, device=DEVICE).normal_(0.0, 1.0, generator=g)
        keys = [x[:, 7 * H * D:8 * H * D].view(tokens, H, D) for x in wide.unbind(0)]
        values = [x[:, 8 * H * D:].view(tokens, H, D) for x in wide.unbind(0)]
    else:
        both = torch.empty((2, L, tokens, H, D), dtype=dt, device=DEVICE).normal_(0.0, 1.0, generator=g)
        keys, values = list(both[0].unbind(0)), list(both[1].unbind(0))
    state = {"case": case, "keys": keys, "values": values, "slots": slots, "tables": tables, "contexts": contexts,
             "lengths": lengths, "tokens": tokens, "scales": [(None, None)] * L}
    if case["cache"] != "auto":
        scales = torch.empty((L, 2, 1), device=DEVICE).uniform_(0.01, 0.1, generator=g)
        state["scales"] = [(s[0], s[1]) for s in scales.unbind(0)]
    if case["layout"] == "flash":
        whole, layers = _pool(case, cache_dt, g)
        state.update(caches=[(p[0], p[1]) for p in layers], out=whole, write=cache_ops.reshape_and_cache_flash)
    else:
        x = 16 // torch.empty((), dtype=cache_dt).element_size()
        kc = _filled((L, NB, H, D // x, bs, x), cache_dt, g)
        vc = _filled((L, NB, H, D, bs), cache_dt, g)
        state.update(caches=list(zip(kc.unbind(0), vc.unbind(0))), out=(kc, vc), write=cache_ops.reshape_and_cache)
    return state


def _prepare_transfer(case, g, host):
    dt = DTYPES[case["dtype"]]
    _, src = _worker(case, dt, g, 0)
    out, dst = _worker(case, torch.bfloat16 if case.get("dequant") else dt, g, 1)
    counts = _block_counts(case)
    sp, dp = (torch.randperm(case["blocks"], generator=host) for _ in range(2))
    tables, at = [], 0
    for n in counts:
        tables.append((sp[at:at + n], dp[at:at + n]))
        at += n
    if case.get("tables") == "device":
        tables = [(a.to(DEVICE), b.to(DEVICE)) for a, b in tables]
    else:
        tables = [(a.tolist(), b.tolist()) for a, b in tables]
    state = {"case": case, "src": src, "dst": dst, "out": out, "tables": tables}
    if case.get("dequant"):
        state["scales"] = torch.empty((2, case["layers"]), device=DEVICE).uniform_(0.01, 0.1, generator=g)
    if case["kind"] == "move":
        manager = KVTransferManager(TransferMethod.CUDA_IPC)
        manager.register_worker(0, src, "prefill")
        manager.register_worker(1, dst, "decoding")
        state["manager"] = manager
    return state


def prepare(case, seed):
    g, host = _generators(seed)
    if case["kind"] == "append":
        return _prepare_append(case, g, host)
    if case["kind"] in ("handoff", "move"):
        return _prepare_transfer(case, g, host)
    if case["kind"] == "copy":
        whole, layers = _pool(case, DTYPES[case["dtype"]], g)
        ids = torch.randperm(case["blocks"], generator=host)[:2 * case["pairs"]]
        return {"case": case, "layers": layers, "out": whole, "mapping": ids.view(2, -1).t().contiguous().to(DEVICE)}
    w = KVWorker(0, DEVICE)
    w.init_vecache()
    names = []
    for i, rows in enumerate(_spread(case["images"], case["least"], case["most"], 0.3)):
        names.append(f"request-{i}")
        w.write_vision_blocks(names[-1], torch.empty((rows, case["hidden"]), dtype=DTYPES[case["dtype"]], device=DEVICE).normal_(generator=g))
    return {"case": case, "worker": w, "names": names}


# ---- one pass ----------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "append":
        slots, mode, write = state["slots"], case["cache"], state["write"]
        if case["tables"]:
            slots = cache_ops.compute_slot_mapping(state["tables"], state["contexts"], state["lengths"], case["block"],
                                                   pad_to=state["tokens"], device=torch.device(DEVICE))
        for key, value, (kc, vc), (ks, vs) in zip(state["keys"], state["values"], state["caches"], state["scales"]):
            write(key, value, kc, vc, slots, mode, ks, vs)
        return state["out"]
    if kind == "handoff":
        src, dst = state["src"], state["dst"]
        buffers = [src.extract_kv_blocks(a) for a, _ in state["tables"]]
        if case["dequant"]:
            ks, vs = state["scales"]
            for (_, b), buf in zip(state["tables"], buffers):
                kv_ops.kv_unpack_dequant_fp8(dst.pool, b, buf, ks, vs)
        else:
            for (_, b), buf in zip(state["tables"], buffers):
                dst.write_kv_blocks(b, buf)
        return state["out"]
    if kind == "move":
        for i, (a, b) in enumerate(state["tables"]):
            if not state["manager"].transfer_kv_cache_sync(f"request-{i}", 0, 1, a, b):
                raise RuntimeError("a transfer failed")
        return state["out"]
    if kind == "copy":
        cache_ops.copy_blocks(state["layers"], state["mapping"])
        return state["out"]
    return state["worker"].gather_vision_embeddings(state["names"])


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "append":
        total = sum(_step_lengths(case))
        width = 2 + (2 if case["cache"] == "auto" else 1)
        return {"bytes": case["layers"] * (total * 2 * _row(case) * width + 8 * total), "flops": 0}
    if kind == "gather":
        return {"bytes": 2 * 2 * case["hidden"] * sum(_spread(case["images"], case["least"], case["most"], 0.3)), "flops": 0}
    chunk = case["block"] * _row(case) * (1 if case["dtype"] == "u8" else 2)
    if kind == "copy":
        return {"bytes": 2 * case["pairs"] * case["layers"] * 2 * chunk, "flops": 0}
    payload = sum(_block_counts(case)) * case["layers"] * 2 * chunk
    if kind == "move":
        return {"bytes": 2 * payload, "flops": 0}
    # a hand-over's buffer is written by the pack and read by the unpack; dequantised values are two bytes
    return {"bytes": payload * (5 if case["dequant"] else 4), "flops": 0}


def tolerance(case):
    return "exact"
