"""Performance cases: the work a user of this package gives it, through its public entry points.

Three kinds of work, each over the sizes it meets in use:

* ``pipeline`` -- ``KVSSDPipeline.decode`` of one query over a layer kept in HBM or in page-locked host memory;
* ``decode``   -- the hip backend over a packed batch: a prepared decode (what a loop over a model's layers keeps)
  or one ``run`` call, with or without a block table, for every head size, group size, block size and GQA ratio;
* ``gather``, ``encode``, ``vllm`` -- the record codec on the GPU: records into packed arrays with their checks,
  keys and values into records, and a vLLM block to its record and back.

Keys, values and queries are Gaussian (INT2 ones with 5 % outliers, as the benchmark's), quantised here by a plain
torch restatement of the codec, so that ``exact`` shares no code with the package.
"""

from __future__ import annotations

import math
import sys
import tempfile
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT / "kvssd-attention_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "kvssd-attention_amd"))

from kvssd import CacheSpec, KVCacheStore, KVSSDPipeline, RecentSinkBlocks  # noqa: E402
from kvssd.backends import PackedBatch, resolve_attention_backend  # noqa: E402
from kvssd.records_hip import encode_records, gather_records  # noqa: E402
from kvssd.vllm_codec_hip import decode_vllm_block, encode_vllm_block  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
CHUNK = 16384  # tokens made or dequantised at a time


def _decode(name, tokens, bits, qh, kvh, d, g, bt, dtype="f16", select=0, entry="prepared"):
    return dict(name=name, kind="decode", tokens=tokens, bits=bits, qh=qh, kvh=kvh, d=d, g=g, bt=bt, dtype=dtype,
                select=select, entry=entry)


def listed():
    return [
        # the shortest context of the benchmark, one layer in HBM, through the pipeline: launches and host work
        dict(name="pipeline_hbm_4k", kind="pipeline", where="hbm", tokens=4096, bits=4, qh=32, kvh=8, d=128, g=32, bt=128,
             dtype="f16", sink=0, recent=0),
        # a layer in page-locked host memory, streamed over PCIe in the pipeline's default 4-block chunks
        dict(name="pipeline_host_16k", kind="pipeline", where="host", tokens=16384, bits=4, qh=32, kvh=8, d=128, g=32,
             bt=128, dtype="f16", sink=0, recent=0),
        # long contexts of the benchmark's model shape, the last block partly filled
        _decode("decode_int4_128k", 131072 - 51, 4, 32, 8, 128, 32, 128),
        _decode("decode_int2_128k", 131072, 2, 32, 8, 128, 32, 128, dtype="bf16"),
        _decode("decode_int4_1m", 1048576, 4, 32, 8, 128, 32, 128),
        # sink + recent blocks of a 256K context, 8 query heads per kv head
        _decode("decode_sparse_gqa8", 262144, 4, 64, 8, 128, 32, 128, select=33),
        # small head size (one run call over a fresh batch, no kept plan)
        _decode("decode_d64_run_16k", 16384 - 7, 4, 32, 8, 64, 32, 128, entry="run"),
        # pages of 32 tokens in table order, half of the cache attended
        _decode("decode_page32_32k", 65536, 4, 32, 8, 128, 32, 32, select=1024),
        # large head size, groups of 64, bfloat16, 6 query heads per kv head
        _decode("decode_d256_g64_24k", 24576 + 33, 4, 24, 4, 256, 64, 64, dtype="bf16"),
        # one 128K layer's records into the packed arrays (every record checked)
        dict(name="gather_int4_128k", kind="gather", tokens=131072, bits=4, kvh=8, d=128, g=32, bt=128),
        # one layer's keys and values into records, the last block padded
        dict(name="encode_int4_128k", kind="encode", tokens=131072 - 77, bits=4, kvh=8, d=128, g=32, bt=128, dtype="bf16"),
        # a 64-token vLLM block of 32 layers (8 kv heads, head_dim 128, K and V) to its record and back
        dict(name="vllm_block_8m", kind="vllm", elements=8388608, bits=4, g=32, dtype="f16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pipeline", "decode", "decode", "general", "general", "general", "gather", "encode", "vllm"])
    bits = rng.choice([4, 4, 2])
    dtype = rng.choice(["f16", "bf16", "f32"])
    if kind == "pipeline":
        where = rng.choice(["hbm", "host"])
        recent = rng.choice([0, rng.randint(4, 40)])
        return dict(kind="pipeline", where=where, tokens=_log_int(rng, 300, 131072 if where == "hbm" else 16384), bits=bits,
                    qh=8 * rng.choice([1, 4, 8]), kvh=8, d=128, g=32, bt=128, dtype=dtype, sink=1 if recent else 0,
                    recent=recent)
    if kind == "decode":
        # the matrix-core shapes: head_dim 128, groups of 32, whole 128-token sub-blocks
        kvh, bt = rng.choice([2, 4, 8, 8, 8]), rng.choice([128, 128, 256])
        tokens = _log_int(rng, 500, 524288)
        blocks = -(-tokens // bt)
        select = rng.choice([0, 0, rng.randint(1, blocks)])
        return dict(kind="decode", tokens=tokens, bits=bits, qh=kvh * rng.choice([1, 2, 4, 5, 8]), kvh=kvh, d=128, g=32,
                    bt=bt, dtype=dtype, select=select, entry=rng.choice(["prepared", "run"]))
    if kind == "general":
        # every other shape: head and group sizes, small pages, wide GQA, multi-query
        d = rng.choice([64, 64, 96, 128, 128, 256])
        g = rng.choice([x for x in (16, 32, 32, 64, 128) if d % x == 0])
        bt = rng.choice([16, 32, 64, 128])
        kvh = rng.choice([1, 2, 4, 8])
        tokens = _log_int(rng, 200, 32768)
        blocks = -(-tokens // bt)
        select = rng.choice([0, 0, rng.randint(1, blocks)])
        return dict(kind="decode", tokens=tokens, bits=bits, qh=kvh * rng.choice([1, 4, 6, 8, 12, 16]), kvh=kvh, d=d, g=g,
                    bt=bt, dtype=dtype, select=select, entry=rng.choice(["prepared", "run"]))
    d = rng.choice([64, 128, 128, 256])
    if kind in ("gather", "encode"):
        return dict(kind=kind, tokens=_log_int(rng, 100, 131072), bits=bits, kvh=rng.choice([1, 4, 8, 8]), d=d,
                    g=rng.choice([32, 32, 64]), bt=rng.choice([32, 128, 128]), **({} if kind == "gather" else {"dtype": dtype}))
    return dict(kind="vllm", elements=128 * _log_int(rng, 16, 65536), bits=bits, g=rng.choice([32, 64]), dtype=dtype)


# --------------------------------------------------------------------------- inputs


def _quantise(x, bits, g):
    """(packed uint8, fp16 scales) of groups of ``g`` along the last dimension, codes low bits first."""
    mid = 1 << (bits - 1)
    groups = x.float().reshape(*x.shape[:-1], x.shape[-1] // g, g)
    # divided by a tensor: by a plain number a GPU multiplies with its reciprocal, which rounds differently
    amax = groups.abs().amax(dim=-1).clamp_min(1e-8)
    scale = amax / torch.full_like(amax, mid - 1)
    codes = (torch.round(groups / scale.unsqueeze(-1)).clamp(-mid, mid - 1) + mid).to(torch.uint8).reshape(x.shape)
    per = 8 // bits
    lanes = codes.reshape(*x.shape[:-1], -1, per)
    packed = lanes[..., 0].clone()
    for i in range(1, per):
        packed |= lanes[..., i] << (i * bits)
    return packed, scale.to(torch.float16)


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * seed + 7)


def _values(gen, shape, dtype, bits):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    if bits == 2:
        x = torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.05, 8 * x, x)
    return x.to(dtype)


def _query(gen, case):
    # scaled scores of standard deviation 2: attention that picks out some tokens, as a trained model's does
    q = 2 * torch.randn((case["qh"], case["d"]), generator=gen, device="cuda", dtype=torch.float32)
    return q.to(DTYPES[case["dtype"]])


def _blocks(case):
    return -(-case["tokens"] // case["bt"])


def _valid(case):
    nb, bt = _blocks(case), case["bt"]
    valid = torch.full((nb,), bt, dtype=torch.int32)
    valid[-1] = case["tokens"] - (nb - 1) * bt
    return valid


def _packed_arrays(case, seed):
    """K and V of a layer as packed arrays [blocks, bt, kvh, ...]; tokens past the end are zeros."""
    gen = _generator(seed)
    nb, bt, kvh, d, g, bits = _blocks(case), case["bt"], case["kvh"], case["d"], case["g"], case["bits"]
    out = []
    for _ in range(2):
        packed = torch.empty((nb * bt, kvh, d * bits // 8), dtype=torch.uint8, device="cuda")
        scales = torch.empty((nb * bt, kvh, d // g), dtype=torch.float16, device="cuda")
        for a in range(0, nb * bt, CHUNK):
            n = min(CHUNK, nb * bt - a)
            x = _values(gen, (n, kvh, d), torch.float16, bits)
            if a + n > case["tokens"]:
                x[max(case["tokens"] - a, 0):] = 0
            packed[a:a + n], scales[a:a + n] = _quantise(x, bits, g)
        out.append((packed.view(nb, bt, kvh, -1), scales.view(nb, bt, kvh, -1)))
    query = _query(gen, case)
    table = None
    if case["select"]:
        # the cache's first block, then the most recent ones; a longer selection is spread over the cache
        n = case["select"]
        if 16 * n <= nb:
            ids = [0] + list(range(nb - n + 1, nb))
        else:
            ids = sorted(torch.randperm(nb, generator=torch.Generator().manual_seed(seed))[:n].tolist())
        table = torch.tensor(ids[:n], dtype=torch.int32)
    return query, out[0], out[1], table


def _layer(case, seed):
    """Keys, values [tokens, kvh, d] and a query."""
    gen = _generator(seed)
    dtype = DTYPES[case.get("dtype", "f16")]
    shape = (case["tokens"], case["kvh"], case["d"])
    keys = _values(gen, shape, dtype, case["bits"])
    values = _values(gen, shape, dtype, case["bits"])
    return keys, values, _query(gen, case) if "qh" in case else None


def _spec(case):
    return CacheSpec(1, case["kvh"], case["d"], case["bt"], case["bits"], case["g"])


def _scale(case):
    return 1.0 / math.sqrt(case["d"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pipeline":
        keys, values, query = _layer(case, seed)
        with tempfile.TemporaryDirectory(prefix="kvssd_cases_") as root:
            store = KVCacheStore.create(root, keys[None], values[None], _spec(case))
            pipe = KVSSDPipeline(store, device="cuda", attention_backend="hip")
            if case["where"] == "hbm":
                pipe.load_resident()
            else:
                pipe.load_host_resident()
        selector = RecentSinkBlocks(case["sink"], case["recent"]) if case["recent"] else None
        return dict(case=case, pipe=pipe, query=query, selector=selector)
    if kind == "decode":
        query, (pk, sk), (pv, sv), table = _packed_arrays(case, seed)
        batch = PackedBatch(pk, pv, sk, sv, _valid(case).cuda(), case["bits"], case["g"])
        backend = resolve_attention_backend("hip", query.device)
        table = None if table is None else table.cuda()
        state = dict(case=case, backend=backend, query=query, batch=batch, table=table)
        if case["entry"] == "prepared":
            state["prepared"] = backend.prepare(query, batch, _scale(case), table)
        return state
    if kind == "gather":
        keys, values, _ = _layer(case, seed)
        spec = _spec(case)
        raw = encode_records(keys, values, spec, 0)[0].view(-1)
        return dict(case=case, raw=raw, spec=spec, count=_blocks(case))
    if kind == "encode":
        keys, values, _ = _layer(case, seed)
        return dict(case=case, keys=keys, values=values, spec=_spec(case))
    dtype = DTYPES[case["dtype"]]
    values = _values(_generator(seed), (case["elements"],), dtype, case["bits"])
    return dict(case=case, values=values, destination=torch.empty_like(values))


# --------------------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "pipeline":
        return state["pipe"].decode(state["query"], 0, state["selector"])
    if kind == "decode":
        if case["entry"] == "prepared":
            return state["prepared"](state["query"])
        return state["backend"].run(state["query"], state["batch"], _scale(case), state["table"])
    if kind == "gather":
        return gather_records(state["raw"], state["spec"], state["count"])
    if kind == "encode":
        return encode_records(state["keys"], state["values"], state["spec"], 0)
    record = encode_vllm_block(state["values"], bits=case["bits"], group_size=case["g"])
    decode_vllm_block(record, state["destination"])
    return record, state["destination"]


# --------------------------------------------------------------------------- work, tolerance, exact results


def _attended(case):
    """Tokens one pass attends over."""
    nb, bt = _blocks(case), case["bt"]
    if case["kind"] == "pipeline":
        return min(case["tokens"], (case["sink"] + case["recent"]) * bt) if case["recent"] else case["tokens"]
    return min(case["tokens"], case["select"] * bt) if case["select"] else case["tokens"]


def work(case):
    kind, bits = case["kind"], case["bits"]
    if kind == "vllm":
        item = 4 if case["dtype"] == "f32" else 2
        n = case["elements"]
        record = n * bits // 8 + 2 * n // case["g"]
        return {"bytes": 2 * (n * item + record), "flops": 6 * n}
    d, kvh, g = case["d"], case["kvh"], case["g"]
    per_token = kvh * (2 * d * bits // 8 + 4 * (d // g))  # packed K and V with their scales
    if kind in ("pipeline", "decode"):
        n = _attended(case)
        return {"bytes": n * per_token + 6 * case["qh"] * d, "flops": 4 * case["qh"] * d * n}
    n = _blocks(case) * case["bt"]
    if kind == "gather":
        return {"bytes": 2 * n * per_token, "flops": 0}
    item = 4 if case["dtype"] == "f32" else 2
    return {"bytes": 2 * case["tokens"] * kvh * d * item + n * per_token, "flops": 6 * case["tokens"] * kvh * d}


def tolerance(case):
    if case["kind"] not in ("pipeline", "decode"):
        return "exact"
    # softmax weights times value scales are rounded to 16 bits, and the codes' offset is taken out of 32-bit sums,
    # whose share of the result grows with the number of tokens averaged (2.5e-4 seen at 128K tokens, 9.5e-4 at 1M)
    matrix = 1e-3 * max(1.0, _attended(case) / 262144)
    if case["kind"] == "pipeline":
        # the result is stored in the query's type (fp16: 2.3e-4 seen)
        return {"rel": {"f16": 1e-3, "bf16": 7e-3, "f32": matrix}[case["dtype"]]}
    if case["d"] == 128 and case["g"] == 32 and case["bt"] % 128 == 0 and case["qh"] // case["kvh"] <= 8:
        return {"rel": matrix}
    return {"rel": 1e-5}  # 32-bit sums throughout


def _dequantised(packed, scales, bits, g):
    """[tokens, kvh, d] in 64 bits."""
    per = 8 // bits
    codes = torch.stack([(packed >> (bits * i)) & ((1 << bits) - 1) for i in range(per)], dim=-1)
    codes = codes.reshape(*packed.shape[:-1], -1).double() - (1 << (bits - 1))
    return codes * scales.double().repeat_interleave(g, dim=-1)


def _attention(query, k, v, rows, case):
    """Softmax attention of ``query`` over the token rows ``rows`` of packed K and V, in 64 bits."""
    (pk, sk), (pv, sv) = k, v
    kvh, d, bits, g = case["kvh"], case["d"], case["bits"], case["g"]
    q = query.double().view(kvh, -1, d)
    spans = [rows[a:a + CHUNK] for a in range(0, len(rows), CHUNK)]
    scores = torch.cat(
        [torch.matmul(q, _dequantised(pk[r], sk[r], bits, g).permute(1, 2, 0).contiguous()) for r in spans], dim=-1
    ) * _scale(case)
    lse = torch.logsumexp(scores, dim=-1)
    weights = torch.exp(scores - lse.unsqueeze(-1))
    out = torch.zeros_like(q)
    for i, r in enumerate(spans):
        w = weights[..., i * CHUNK:i * CHUNK + len(r)].contiguous()
        out += torch.matmul(w, _dequantised(pv[r], sv[r], bits, g).permute(1, 0, 2).contiguous())
    return out.view(-1, d), lse.view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        query, k, v, table = _packed_arrays(case, seed)
        flat = [tuple(t.flatten(0, 1) for t in pair) for pair in (k, v)]
        valid = _valid(case).cuda()
        ids = torch.arange(_blocks(case), device="cuda") if table is None else table.cuda().long()
        rows = ids[:, None] * case["bt"] + torch.arange(case["bt"], device="cuda")
        rows = rows[torch.arange(case["bt"], device="cuda") < valid[ids][:, None]]
        return _attention(query, flat[0], flat[1], rows, case)
    if kind == "pipeline":
        keys, values, query = _layer(case, seed)
        k, v = _quantise(keys, case["bits"], case["g"]), _quantise(values, case["bits"], case["g"])
        nb, bt = _blocks(case), case["bt"]
        ids = range(nb)
        if case["recent"]:
            ids = sorted(set(range(min(case["sink"], nb))) | set(range(max(nb - case["recent"], 0), nb)))
        rows = torch.cat([torch.arange(b * bt, min((b + 1) * bt, case["tokens"])) for b in ids]).cuda()
        return _attention(query, k, v, rows, case)[0]
    if kind == "vllm":
        values = _values(_generator(seed), (case["elements"],), DTYPES[case["dtype"]], case["bits"])
        packed, scales = _quantise(values.view(-1, case["g"]), case["bits"], case["g"])
        flat = _dequantised(packed.unsqueeze(1), scales.unsqueeze(1), case["bits"], case["g"])
        return None, flat.view(-1)
    return None
