"""Work that programs have this operator do, as cases to time and compare.

A case is a dict of plain values; ``prepare`` makes the tensors and the plan a
serving program holds before a call, ``run`` is one pass through the public
entry points (``DecodePlan``, ``append_kv``), ``exact`` the same result in 64
bits from plain torch. Four kinds of pass:

* ``decode``: one ``plan.run`` over a batch, launched eagerly;
* ``step``: one token's attention in a model of ``layers`` layers, captured in
  a graph by the program: per layer the new token's K and V rows are written
  into the paged cache, the layer is decoded and its output cast to the
  model's type;
* ``csr``: a scheduler keeps its page lists on the GPU in CSR form, so each
  pass loads them (``refresh_csr``) and decodes;
* ``append``: a prompt's K and V rows are written into the paged cache.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "paged-decode-lab_amd"))

from paged_decode.csr import paged_csr  # noqa: E402
from paged_decode.layout import Layout  # noqa: E402
from paged_decode.runtime import DecodePlan, append_kv  # noqa: E402

# fmt -> (q type, K/V type)
_TYPES = {
    "f32": (torch.float32, torch.float32),
    "f16": (torch.float16, torch.float16),
    "bf16": (torch.bfloat16, torch.bfloat16),
    "e4m3": (torch.float16, torch.float8_e4m3fn),
    "e5m2": (torch.float16, torch.float8_e5m2),
    "bf16_e4m3": (torch.bfloat16, torch.float8_e4m3fn),
}

# What a case holds unless it says otherwise: 32 query and 8 KV heads of 128
# dims (Llama-3-8B), pages of 16 tokens, partitions of 256.
_DEFAULTS = {"kind": "decode", "fmt": "f16", "batch": 4, "q_heads": 32, "kv_heads": 8, "dim": 128, "page": 16,
             "context": 4096, "lengths": "uniform", "shared": 0.0, "reserve": 1, "split": 256, "merge": "serial",
             "heavy": 0.0, "layers": 1, "tokens": 1}


def listed():
    return [
        # The smallest call: the FP32 check that the reference's tests and this repository's named workloads run.
        {"name": "f32_b2_l256", "fmt": "f32", "batch": 2, "q_heads": 8, "kv_heads": 2, "dim": 64, "context": 256,
         "lengths": "ragged"},
        # The headline: a small batch of 4K contexts, launched eagerly.
        {"name": "f16_b4_l4096", "batch": 4},
        # One user's token through 32 layers, captured in a graph, with room reserved for the tokens to come.
        {"name": "step_bf16_b1_l4096", "kind": "step", "fmt": "bf16", "batch": 1, "layers": 32, "reserve": 2},
        # A quantized cache at a serving batch, contexts of all ages.
        {"name": "e4m3_b16_l4096", "fmt": "e4m3", "batch": 16, "lengths": "ragged"},
        # A large serving batch with long, uneven contexts on 32-token pages: the largest decode.
        {"name": "bf16_b64_l8192", "fmt": "bf16", "batch": 64, "page": 32, "context": 8192, "lengths": "ragged"},
        # Many short chats at once: every row is small.
        {"name": "f16_b256_l256", "batch": 256, "context": 256, "lengths": "ragged"},
        # Multi-query heads at a large batch, 5% of the keys scaled up.
        {"name": "mqa_b128_l1024", "batch": 128, "q_heads": 16, "kv_heads": 1, "dim": 64, "context": 1024,
         "heavy": 0.05},
        # One long document, multi-head attention.
        {"name": "mha_b1_l32768", "batch": 1, "kv_heads": 32, "context": 32768, "split": 512},
        # Continuations of one prompt, contexts from empty to 8K, a quarter of the pages shared.
        {"name": "shared_b16_l8192", "batch": 16, "page": 32, "context": 8192, "lengths": "wide", "shared": 0.25,
         "split": 128},
        # FP32 inputs at serving size: the precise path.
        {"name": "f32_b8_l4096", "fmt": "f32", "batch": 8, "lengths": "ragged"},
        # Page lists kept on the GPU by the scheduler, twice the longest context reserved.
        {"name": "csr_bf16_b32_l4096", "kind": "csr", "fmt": "bf16", "batch": 32, "lengths": "ragged", "reserve": 2},
        # Prompts written into the cache before their first decode.
        {"name": "append_bf16_b8_t1024", "kind": "append", "fmt": "bf16", "batch": 8, "tokens": 1024},
    ]


_HEADS = [(32, 8, 128), (32, 8, 64), (32, 4, 128), (32, 2, 128), (28, 4, 128), (40, 8, 128), (8, 2, 64), (16, 1, 64),
          (16, 16, 128), (32, 32, 128), (24, 3, 128), (64, 8, 128)]


def draw(rng):
    """One more case: any head layout, type and page size, batches of 1 to 256, contexts of 17 to 32768 tokens."""
    while True:
        q_heads, kv_heads, dim = rng.choice(_HEADS)
        case = {"kind": rng.choice(["decode"] * 7 + ["step", "csr", "append"]),
                "fmt": rng.choice(["f16", "f16", "bf16", "bf16", "e4m3", "e5m2", "bf16_e4m3", "f32"]),
                "batch": int(round(2 ** rng.uniform(0, 8))), "q_heads": q_heads, "kv_heads": kv_heads, "dim": dim,
                "page": rng.choice([16, 32]), "context": int(round(math.exp(rng.uniform(math.log(17), math.log(32768))))),
                "lengths": rng.choice(["uniform", "ragged", "ragged", "wide"]), "split": rng.choice([128, 256, 256, 512]),
                "merge": rng.choice(["serial", "serial", "shared"])}
        if case["kind"] == "decode":
            case["shared"] = rng.choice([0.0, 0.0, 0.0, 0.25, 0.5])
            case["reserve"] = rng.choice([1, 1, 2])
        elif case["kind"] == "step":
            case["layers"] = rng.choice([2, 4, 8])
            case["reserve"] = rng.choice([1, 2])
        elif case["kind"] == "csr":
            case["reserve"] = rng.choice([1, 2])
        else:
            case["tokens"] = min(case["context"], int(round(2 ** rng.uniform(0, 11))))
            case["lengths"] = "uniform"
        full = _full(case)
        cache = (full["layers"] * full["batch"] * full["context"] * full["reserve"] * 2 * kv_heads * dim
                 * _TYPES[full["fmt"]][1].itemsize)
        if 1 << 17 <= cache <= 3 << 28 and work(case)["bytes"] <= 7e8:
            return case


def _full(case):
    return {**_DEFAULTS, **case}


def _lengths(c, rng):
    n = np.full(c["batch"], c["context"], dtype=np.int32)
    if c["lengths"] == "ragged":  # a quarter of the context to all of it
        n[1:] = rng.integers(max(1, c["context"] // 4), c["context"] + 1, size=c["batch"] - 1)
        if c["batch"] == 1:
            n[0] = c["context"]
    elif c["lengths"] == "wide":  # empty to full
        n[1:] = rng.integers(0, c["context"] + 1, size=c["batch"] - 1)
    return n


def _metadata(c, seed):
    """Layout, page table and lengths; the shared pages are the rows' leading ones. ``reserve`` widens the table."""
    # The lengths are the case's own, so that each seed's pass is the same amount of work.
    lengths = _lengths(c, np.random.default_rng(c["batch"] * 65537 + c["context"]))
    rng = np.random.default_rng(seed)
    width = -(-c["context"] * c["reserve"] // c["page"])
    shared = int(-(-c["context"] // c["page"]) * c["shared"])
    own = width - shared
    pages = shared + c["batch"] * own
    ids = rng.permutation(pages).astype(np.int32)
    table = np.empty((c["batch"], width), dtype=np.int32)
    table[:, :shared] = ids[:shared]
    table[:, shared:] = ids[shared:].reshape(c["batch"], own)
    if c["reserve"] == 1:
        for b, n in enumerate(lengths):
            table[b, -(-int(n) // c["page"]):] = -1
    return Layout(c["batch"], c["q_heads"], c["kv_heads"], c["dim"], c["page"], pages), table, lengths


def _values(shape, dtype, gen, heavy=0.0):
    """N(0, 1) values in the stored type with their scale (1 for unquantized types)."""
    if dtype.itemsize > 1:
        x = torch.randn(shape, device="cuda", dtype=dtype, generator=gen)
        if heavy:
            x.mul_(torch.where(torch.rand(shape, device="cuda", generator=gen) < heavy, 20.0, 1.0).to(dtype))
        return x, 1.0
    x = torch.randn(shape, device="cuda", dtype=torch.float16, generator=gen)
    scale = 5.5 / float(torch.finfo(dtype).max)  # a calibrated scale, as a checkpoint carries it
    return x.div_(scale).clamp_(-float(torch.finfo(dtype).max), float(torch.finfo(dtype).max)).to(dtype), scale


def prepare(case, seed):
    c = _full(case)
    q_type, kv_type = _TYPES[c["fmt"]]
    layout, table, lengths = _metadata(c, seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cache_shape = (layout.physical_pages, c["page"], c["kv_heads"], c["dim"])
    s = {"case": c, "layout": layout, "table": table, "lengths": lengths}
    if c["kind"] == "append":
        s["k"] = torch.zeros(cache_shape, device="cuda", dtype=kv_type)
        s["v"] = torch.zeros(cache_shape, device="cuda", dtype=kv_type)
        new = (c["batch"], c["tokens"], c["kv_heads"], c["dim"])
        s["k_new"], s["v_new"] = _values(new, kv_type, gen)[0], _values(new, kv_type, gen)[0]
        s["d_table"] = torch.from_numpy(table).cuda()
        s["positions"] = torch.from_numpy((lengths - c["tokens"]).astype(np.int32)).cuda()
        return s
    layers = c["layers"]
    s["q"] = torch.randn((layers, c["batch"], c["q_heads"], c["dim"]), device="cuda", dtype=q_type, generator=gen)
    s["cache"], s["scale"] = _values((layers, 2, *cache_shape), kv_type, gen, c["heavy"])
    s["plan"] = DecodePlan(layout, table, lengths, split_tokens=c["split"], merge=c["merge"],
                           max_context=min(c["context"] * c["reserve"], table.shape[1] * c["page"]))
    if c["kind"] == "csr":
        live = lengths > 0
        indptr, indices, last = paged_csr(Layout(int(live.sum()), *list(vars(layout).values())[1:]), table[live],
                                          lengths[live])
        counts = np.zeros(c["batch"], dtype=np.int64)  # an empty context is an empty list
        counts[live] = np.diff(np.asarray(indptr))
        last_all = np.zeros(c["batch"], dtype=np.int32)
        last_all[live] = np.asarray(last)
        s["indptr"] = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).cuda()
        s["indices"] = torch.from_numpy(np.asarray(indices, dtype=np.int32)).cuda()
        s["last"] = torch.from_numpy(last_all).cuda()
    elif c["kind"] == "step":
        new = (layers, 2, c["batch"], 1, c["kv_heads"], c["dim"])
        s["new"] = _values(new, kv_type, gen)[0]
        s["d_table"] = torch.from_numpy(table).cuda()
        s["positions"] = torch.from_numpy(np.maximum(lengths - 1, 0).astype(np.int32)).cuda()
        s["out"] = torch.empty((layers, c["batch"], c["q_heads"], c["dim"]), device="cuda",
                               dtype=torch.float32 if kv_type == torch.float32 else q_type)
        _step(s)  # once outside the capture, as a program warms up
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
    return s


def _step(s):
    for i in range(s["case"]["layers"]):
        k, v = s["cache"][i, 0], s["cache"][i, 1]
        append_kv(s["layout"], k, v, s["d_table"], s["positions"], s["new"][i, 0], s["new"][i, 1])
        s["out"][i].copy_(s["plan"].run(s["q"][i], k, v, k_scale=s["scale"], v_scale=s["scale"]))


def run(state):
    s = state
    kind = s["case"]["kind"]
    if kind == "append":
        append_kv(s["layout"], s["k"], s["v"], s["d_table"], s["positions"], s["k_new"], s["v_new"])
        return s["k"], s["v"]
    if kind == "step":
        s["graph"].replay()
        return s["out"], s["cache"]
    if kind == "csr":
        s["plan"].refresh_csr(s["indptr"], s["indices"], s["last"])
    return s["plan"].run(s["q"][0], s["cache"][0, 0], s["cache"][0, 1], k_scale=s["scale"], v_scale=s["scale"])


def work(case):
    c = _full(case)
    kv = _TYPES[c["fmt"]][1].itemsize
    row = c["kv_heads"] * c["dim"] * kv  # one token's K, or V
    if c["kind"] == "append":
        return {"bytes": 4 * c["batch"] * c["tokens"] * row, "flops": 0}
    lengths = _lengths(c, np.random.default_rng(c["batch"] * 65537 + c["context"])).astype(np.int64)
    shared = int(-(-c["context"] // c["page"]) * c["shared"]) * c["page"]
    once = int(np.minimum(lengths, shared).max(initial=0) + np.maximum(lengths - shared, 0).sum())  # tokens stored
    q = c["batch"] * c["q_heads"] * c["dim"]
    out = q * (4 + _TYPES[c["fmt"]][0].itemsize)
    table = 4 * int((-(-lengths // c["page"])).sum())
    new = 4 * c["batch"] * row if c["kind"] == "step" else 0
    return {"bytes": c["layers"] * (2 * once * row + out + table + new),
            "flops": c["layers"] * 4 * int(lengths.sum()) * c["q_heads"] * c["dim"]}


def tolerance(case):
    c = _full(case)
    if c["kind"] == "append":
        return "exact"
    # About four times the error that these paths show against 64 bits: 2.4e-6 where the weights are split into two
    # bfloat16 parts, up to 4.1e-7 otherwise, and a step's cast to the model's type (1.7e-3, 2.1e-4) on top.
    bf16 = _TYPES[c["fmt"]][0] == torch.bfloat16
    if c["kind"] == "step" and c["fmt"] != "f32":
        return {"rel": 7e-3 if bf16 else 9e-4}
    return {"rel": 1e-5 if bf16 else 3e-6}


def _rows_of(pages, rows):
    return pages.view(torch.uint8)[rows].view(pages.dtype) if pages.dtype.itemsize == 1 else pages[rows]


def exact(case, seed):
    c = _full(case)
    s = prepare({**case, "kind": "decode"} if c["kind"] == "csr" else case, seed)
    if c["kind"] == "append":
        k, v = s["k"].double(), s["v"].double()
        for b in range(c["batch"]):
            pos = torch.arange(c["tokens"], device="cuda") + int(s["lengths"][b]) - c["tokens"]
            page = s["d_table"][b].long()[pos // c["page"]]
            k[page, pos % c["page"]] = s["k_new"][b].double()
            v[page, pos % c["page"]] = s["v_new"][b].double()
        return k, v
    table = torch.from_numpy(s["table"]).long().cuda()
    cache = s["cache"]
    if c["kind"] == "step":
        cache = cache.double()
        for b in range(c["batch"]):
            at = max(int(s["lengths"][b]) - 1, 0)
            page = int(s["table"][b, at // c["page"]])
            if page >= 0:
                cache[:, :, page, at % c["page"]] = s["new"][:, :, b, 0].double()
    group = c["q_heads"] // c["kv_heads"]
    out = torch.zeros(s["q"].shape, device="cuda", dtype=torch.float64)
    for i in range(c["layers"]):
        for b, n in enumerate(int(x) for x in s["lengths"]):
            if n == 0:
                continue
            rows = table[b, :-(-n // c["page"])]
            # [Hkv, tokens, D]
            k, v = (_rows_of(cache[i, j], rows).reshape(-1, c["kv_heads"], c["dim"])[:n].double().transpose(0, 1)
                    .contiguous() for j in (0, 1))
            q = s["q"][i, b].double().view(c["kv_heads"], group, c["dim"])
            scores = torch.matmul(q, (k * s["scale"]).transpose(1, 2).contiguous()) / math.sqrt(c["dim"])
            out[i, b] = torch.matmul(torch.softmax(scores, -1), v * s["scale"]).reshape(c["q_heads"], c["dim"])
    return (out, cache) if c["kind"] == "step" else out[0]
