"""The work that a user of this framework has it do, as measurable cases.

One case is one call, or one layer-step, of the DSA KV-offload decode chain
through the package's public entry points.  The listed sizes come from this
repository's benchmark (``bench.py``), its configurations
(``nanovllm_amd/workloads.py``) and its tests; ``draw`` gives more of the same
ranges: 1 to 64 requests, prompts of 3K to 128K tokens, cache budgets of 2048
to 8192 slots, 4 to 128 attention heads, one or four query rows per request,
bf16 and fp16.

A decode case holds what a serving loop holds: the paged index keys, the slot
pool and HBM caches as the previous step left them, the DRAM caches in
host-mapped memory, and a few steps' index queries that are used in turn, so
that every pass selects anew and copies real misses.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "nanovllm-dsa-offload_amd"))

from nanovllm_amd import dsa_offload_ops as ops  # noqa: E402
from nanovllm_amd.decode_graph import DsaLayerGraph  # noqa: E402
from nanovllm_amd.dsa_indexer_project import dsa_indexer_project, dsa_indexer_project_query_only  # noqa: E402
from nanovllm_amd.host_memory import empty_host_mapped  # noqa: E402
from nanovllm_amd.index_share import CONTEXT_FIELDS, DsaLayerCaches, IndexShareDecodeStep, IndexShareGroupManager  # noqa: E402

BLOCK, TOPK, CKV, KPE, IDX = 128, 2048, 512, 64, 128
ROW_BYTES = 2 * (CKV + KPE)            # one latent KV row
SCALE = 1.0 / math.sqrt(CKV + KPE)
INDEX_HEADS = 32
HIDDEN, RANK = 6144, 2048              # the indexer projection's widths
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}

# Decode steps (LIM, then the miss copy and the attention).
_STEP = {"lo": 32768, "hi": 32768, "cache": 2048, "heads": 64, "mtp": False, "dtype": "bf16", "width": 65536,
         "drift": 0.1, "turns": 2, "short": 0, "layers": 1}


def _step(kind: str, name: str | None = None, **fields) -> dict:
    case = {"kind": kind, **_STEP, **fields}
    return case if name is None else {"name": name, **case}


def listed() -> list[dict]:
    return [
        # One interactive request replayed from a captured decode graph: the smallest step, all latency.
        _step("graph", "graph_step_b1", batch=1, lo=20480, hi=20480),
        # The benchmark's layer-step: 24 requests of 32K, fused copy + attention.
        _step("fused", "fused_step_b24", batch=24),
        # A full mixed batch, prompts of 20K to 64K.
        _step("fused", "fused_step_b64_mixed", batch=64, lo=20480, hi=65536),
        # Speculative verify: four query rows per request, the union of their selections.
        _step("fused", "mtp_step_b16", batch=16, lo=49152, hi=49152, cache=8192, mtp=True),
        # The unfused path of the same chain, an odd batch of ragged fp16 requests, two too short to be offloaded.
        _step("split", "split_step_b13_f16", batch=13, lo=4096, hi=40960, heads=32, dtype="f16", short=2, drift=0.15),
        # A selecting layer and the three layers that share its selection, long prompts.
        _step("share", "indexshare_group_b8", batch=8, lo=65536, hi=65536, layers=4),
        # Selection alone with a large cache budget, where victims are chosen by score.
        _step("lim", "lim_b24_64k_c8192", batch=24, lo=65536, hi=65536, cache=8192, drift=0.65, turns=4),
        # Attention alone, everything cached.
        {"name": "attention_b24", "kind": "attention", "batch": 24, "cache": 2048, "heads": 64, "mtp": False,
         "dtype": "bf16", "short": 0},
        # One rank's share of the heads under tensor parallelism, large cache budget.
        {"name": "copy_attention_b24_h4", "kind": "copy_attention", "batch": 24, "prompt": 65536, "cache": 8192,
         "heads": 4, "misses": 164, "dtype": "bf16"},
        # The projection that makes a decode step's index query and head weights.
        {"name": "indexer_decode_t24", "kind": "indexer_decode", "tokens": 24, "dtype": "bf16"},
        # The same for a prompt's tokens, with the index keys.
        {"name": "indexer_prefill_t4096", "kind": "indexer_prefill", "tokens": 4096, "dtype": "bf16"},
        # A request's first decode: top-C selection and the copy of the chosen rows.
        {"name": "first_decode_32k", "kind": "first_decode", "prompt": 32768, "cache": 2048, "width": 65536,
         "dtype": "bf16"},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("graph", "fused", "fused", "mtp", "split", "share", "lim", "lim_mtp", "attention", "attention",
                       "copy_attention", "indexer_decode", "indexer_prefill", "first_decode"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    heads = rng.choice((4, 8, 16, 32, 64, 64, 128))
    if kind == "indexer_decode":
        return {"kind": kind, "tokens": _log(rng, 1, 256), "dtype": dtype}
    if kind == "indexer_prefill":
        return {"kind": kind, "tokens": _log(rng, 33, 8192), "dtype": dtype}
    if kind == "first_decode":
        prompt = BLOCK * _log(rng, 24, 1024)
        cache = rng.choice([c for c in (2048, 4096, 8192, 2048 + 2 * rng.randrange(1000)) if c <= prompt])
        return {"kind": kind, "prompt": prompt, "cache": cache, "width": max(prompt, 65536), "dtype": dtype}
    if kind == "attention":
        mtp = rng.random() < 0.3
        batch = _log(rng, 1, 16 if mtp else 64)
        return {"kind": kind, "batch": batch, "cache": rng.choice((2048, 2048, 4096, 8192)), "heads": heads, "mtp": mtp,
                "dtype": dtype, "short": rng.randrange(0, 1 + batch // 4)}
    if kind == "copy_attention":
        return {"kind": kind, "batch": _log(rng, 1, 64), "prompt": BLOCK * _log(rng, 64, 128),
                "cache": rng.choice((2048, 4096, 8192)), "heads": heads, "misses": rng.randrange(0, 320), "dtype": dtype}
    mtp = kind in ("mtp", "lim_mtp")
    cache = 8192 if mtp else rng.choice((2048, 2048, 2048, 4096, 8192))
    top = 1024 if kind.startswith("lim") else 512                    # blocks of the longest prompt
    hi = BLOCK * _log(rng, max(24, cache // BLOCK + 1), top)
    lo = max(cache, BLOCK * int(hi / BLOCK * rng.uniform(0.3, 1.0)))
    tokens = 2_000_000 if kind.startswith("lim") else 600_000        # of all requests together
    layers = 1
    if kind == "share":
        layers = rng.choice((2, 3))
        tokens //= layers
    batch = _log(rng, 1, max(1, min(16 if mtp else 64, tokens // hi)))
    return _step({"mtp": "fused", "lim_mtp": "lim"}.get(kind, kind), batch=batch, lo=lo, hi=hi, cache=cache, heads=heads,
                 mtp=mtp, dtype=dtype, width=rng.choice((hi, max(hi, 65536))),
                 drift=round(0.65 if cache > TOPK and not mtp else rng.uniform(0.05, 0.15), 3),
                 turns=4 if cache > TOPK and not mtp else 2, layers=layers,
                 short=rng.randrange(0, 1 + batch // 4) if kind in ("fused", "split") else 0)


# ---------------------------------------------------------------------------
# Inputs.


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _i32(values) -> torch.Tensor:
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _lengths(case: dict) -> tuple[list[int], list[int], list[int]]:
    """Candidate tokens, cache budget and visible length of each request
    (fixed by the case, not by the seed).  Short requests have no cache
    budget and attend densely to what they hold."""
    rng = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    n, c, kv = [], [], []
    for b in range(case["batch"]):
        tail = rng.randrange(4, BLOCK)
        if b < case.get("short", 0):
            n.append(0)
            c.append(0)
            kv.append(rng.randrange(100, 1900))
        else:
            n.append(BLOCK * rng.randint(case["lo"] // BLOCK, case["hi"] // BLOCK) if "lo" in case else 0)
            c.append(case["cache"])
            kv.append(case["cache"] + tail)
    return n, c, kv


def _tables(g, blocks: list[int], width: int) -> tuple[torch.Tensor, int]:
    """Block tables over one shuffled pool of blocks, padded with 0."""
    total = max(1, sum(blocks))
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    table = torch.zeros(len(blocks), width, dtype=torch.int32, device="cuda")
    at = 0
    for b, k in enumerate(blocks):
        table[b, :k] = perm[at:at + k]
        at += k
    return table, total


def _rows(table: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
    ids = ids.long()
    return table.long()[ids // BLOCK] * BLOCK + ids % BLOCK


def _dram(g, blocks: int, dtype) -> tuple[torch.Tensor, torch.Tensor]:
    kv = empty_host_mapped((blocks, BLOCK, CKV), dtype, "cuda")
    rope = empty_host_mapped((blocks, BLOCK, KPE), dtype, "cuda")
    for t in (kv, rope):
        for part in t.split(1024):
            part.copy_(_randn(g, *part.shape, dtype=dtype))
    return kv, rope


def _hbm(g, kv: list[int], dtype) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    blocks = [-(-v // BLOCK) for v in kv]
    table, total = _tables(g, blocks, max(blocks))
    return table, _randn(g, total, BLOCK, 1, CKV, dtype=dtype), _randn(g, total, BLOCK, 1, KPE, dtype=dtype)


def _scores(keys: torch.Tensor, query: torch.Tensor, weights: torch.Tensor) -> torch.Tensor:
    return torch.relu(keys @ query.T.contiguous()) @ weights


def _prepare_step(case: dict, seed: int) -> dict:
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    n, c, kv = _lengths(case)
    B, Q = case["batch"], 4 if case["mtp"] else 1
    blocks, width = [x // BLOCK for x in n], case["width"]
    index_table, total = _tables(g, blocks, width // BLOCK)
    keys = _randn(g, total, BLOCK, 1, IDX, dtype=dtype)
    base = _randn(g, B * Q, INDEX_HEADS, IDX)
    drift = case["drift"]
    queries = [((base + drift * _randn(g, B * Q, INDEX_HEADS, IDX)) / math.sqrt(1 + drift * drift)).to(dtype)
               for _ in range(case["turns"])]
    weights = torch.rand(B * Q, INDEX_HEADS, generator=g, device="cuda").to(dtype)
    pool = torch.full((B + 1, width), -1, dtype=torch.int32, device="cuda")
    entries = torch.randperm(B + 1, generator=g, device="cuda")[:B].to(torch.int32)
    s = {"case": case, "turn": 0, "queries": queries[1:] + queries[:1], "weights": weights, "keys": keys, "pool": pool,
         "num_candidate_tokens": _i32(n), "num_cache_tokens": _i32(c), "req_pool_entries": entries,
         "index_block_table": index_table, "rows": B * Q}
    # The pool and the HBM caches as the last query left them: its best tokens cached, in shuffled slots.
    cached = []
    rows = [int(e) for e in entries.tolist()]
    for b in range(B):
        if n[b] == 0:
            cached.append(None)
            continue
        k = keys.view(-1, IDX)[_rows(index_table[b], torch.arange(n[b], device="cuda"))].float()
        best = _scores(k, queries[0][b * Q].float(), weights[b * Q].float())
        for q in range(b * Q + 1, b * Q + Q):
            best = torch.maximum(best, _scores(k, queries[0][q].float(), weights[q].float()))
        top = torch.topk(best, c[b]).indices
        slots = torch.randperm(c[b], generator=g, device="cuda")
        pool[rows[b], top] = slots.to(torch.int32)
        cached.append((top, slots))
    s["topk_src"] = torch.full((B * Q, 1, TOPK), -1, dtype=torch.int32, device="cuda")
    s["topk_dst"] = torch.full((B * Q, 1, TOPK), -1, dtype=torch.int32, device="cuda")
    s["miss_counts"] = torch.zeros(B, dtype=torch.int32, device="cuda")
    if case["mtp"]:
        s["miss_src"] = torch.full((B, 4 * TOPK), -1, dtype=torch.int32, device="cuda")
        s["miss_dst"] = torch.full((B, 4 * TOPK), -1, dtype=torch.int32, device="cuda")
    if case["kind"] == "lim":
        return s
    dram_table, total = _tables(g, blocks, width // BLOCK)
    s["dram_block_table"] = dram_table
    s["actual_seq_lengths_kv"] = _i32(kv)
    s["actual_seq_lengths_query"] = _i32([Q * (b + 1) for b in range(B)])
    s["layers"] = []
    hbm_table = None
    for _ in range(case["layers"]):
        dkv, drope = _dram(g, total, dtype)
        table, hkv, hrope = _hbm(g, kv, dtype)
        hbm_table = table if hbm_table is None else hbm_table
        for b in range(B):
            if cached[b] is not None:
                src, dst = _rows(dram_table[b], cached[b][0]), _rows(hbm_table[b], cached[b][1])
                hkv.view(-1, CKV)[dst] = dkv.view(-1, CKV)[src]
                hrope.view(-1, KPE)[dst] = drope.view(-1, KPE)[src]
        H = case["heads"]
        s["layers"].append({"hbm_kv": hkv, "hbm_rope": hrope, "dram_kv": dkv, "dram_rope": drope,
                            "query": _randn(g, B * Q, H, CKV, dtype=dtype),
                            "query_rope": _randn(g, B * Q, H, KPE, dtype=dtype),
                            "out": torch.zeros(B * Q, H, CKV, dtype=dtype, device="cuda")})
    s["hbm_block_table"] = hbm_table
    if case["kind"] == "share":
        first = s["layers"][0]
        caches = [DsaLayerCaches(l["hbm_rope"], l["hbm_kv"], l["dram_rope"], l["dram_kv"],
                                 index_key_cache=keys if l is first else None,
                                 cache_slots_pool=pool if l is first else None) for l in s["layers"]]
        types = ["full"] + ["shared"] * (case["layers"] - 1)
        s["stack"] = IndexShareDecodeStep(IndexShareGroupManager(case["layers"], types), caches, mtp=False, fused=True)
    if case["kind"] == "graph":
        l = s["layers"][0]
        s["graph"] = DsaLayerGraph(B, index_key_cache=keys, cache_slots_pool=pool, hbm_k_rope=l["hbm_rope"],
                                   hbm_kv_cache=l["hbm_kv"], dram_k_rope=l["dram_rope"], dram_kv_cache=l["dram_kv"],
                                   hbm_block_columns=width // BLOCK, dram_block_columns=width // BLOCK,
                                   heads=case["heads"], index_heads=INDEX_HEADS, scale=SCALE, mtp=case["mtp"],
                                   dtype=dtype)
        s["graph"].capture()
    return s


def _prepare_attention(case: dict, seed: int) -> dict:
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    mtp = case.get("mtp", False)
    B, Q, H, C = case["batch"], 4 if mtp else 1, case["heads"], case["cache"]
    _, c, kv = _lengths(case)
    table, hkv, hrope = _hbm(g, kv, dtype)
    dst = torch.rand(B * Q, C, generator=g, device="cuda").topk(TOPK).indices.to(torch.int32)
    s = {"case": case, "num_cache_tokens": _i32(c), "actual_seq_lengths_kv": _i32(kv),
         "actual_seq_lengths_query": _i32([Q * (b + 1) for b in range(B)]), "hbm_block_table": table, "hbm_kv": hkv,
         "hbm_rope": hrope, "topk_dst": dst.view(B * Q, 1, TOPK).contiguous(),
         "query": _randn(g, B * Q, H, CKV, dtype=dtype), "query_rope": _randn(g, B * Q, H, KPE, dtype=dtype),
         "out": torch.zeros(B * Q, H, CKV, dtype=dtype, device="cuda")}
    if case["kind"] == "copy_attention":
        blocks = case["prompt"] // BLOCK
        s["dram_block_table"], total = _tables(g, [blocks] * B, blocks)
        s["dram_kv"], s["dram_rope"] = _dram(g, total, dtype)
        src = torch.rand(B, case["prompt"], generator=g, device="cuda").topk(TOPK).indices
        s["topk_src"] = src.to(torch.int32).contiguous()
        m = case["misses"]
        s["miss_counts"] = _i32([m + (7 * b) % 41 - 20 if m >= 20 else m for b in range(B)])
    return s


def _prepare_indexer(case: dict, seed: int) -> dict:
    g, dtype, T = _gen(seed), DTYPES[case["dtype"]], case["tokens"]
    s = {"case": case, "hidden": _randn(g, T, HIDDEN, dtype=dtype), "q_c": _randn(g, T, RANK, dtype=dtype),
         "wq_b": (_randn(g, INDEX_HEADS * IDX, RANK) / math.sqrt(RANK)).to(dtype),
         "q": torch.empty(T, INDEX_HEADS, IDX, dtype=dtype, device="cuda"),
         "w": torch.empty(T, INDEX_HEADS, dtype=dtype, device="cuda")}
    w_proj = _randn(g, INDEX_HEADS, HIDDEN) / math.sqrt(HIDDEN)
    pos = torch.randint(0, 65536, (T, 1), generator=g, device="cuda").double()
    angle = (pos * 10000.0 ** (-torch.arange(KPE // 2, device="cuda").double() / (KPE // 2))).repeat_interleave(2, 1)
    s["cos"], s["sin"] = angle.cos().to(dtype), angle.sin().to(dtype)
    if case["kind"] == "indexer_decode":
        s["w_proj"] = w_proj.to(dtype)     # the decode path keeps the head projection in the activations' type
    else:
        s["w_proj"] = w_proj
        s["wk"] = (_randn(g, IDX, HIDDEN) / math.sqrt(HIDDEN)).to(dtype)
        s["k_norm_weight"] = (1 + 0.1 * _randn(g, IDX)).to(dtype)
        s["k_norm_bias"] = (0.1 * _randn(g, IDX)).to(dtype)
        s["k"] = torch.empty(T, IDX, dtype=dtype, device="cuda")
    return s


def _prepare_first_decode(case: dict, seed: int) -> dict:
    g, dtype = _gen(seed), DTYPES[case["dtype"]]
    blocks, cols = case["prompt"] // BLOCK, case["width"] // BLOCK
    index_table, total = _tables(g, [blocks], cols)
    dram_table, _ = _tables(g, [blocks], cols)
    table, hkv, hrope = _hbm(g, [case["cache"] + BLOCK], dtype)
    dkv, drope = _dram(g, total, dtype)
    return {"case": case, "hbm_kv": hkv, "hbm_rope": hrope,
            "pool": torch.full((2, case["width"]), -1, dtype=torch.int32, device="cuda"),
            "args": dict(query=_randn(g, INDEX_HEADS, IDX, dtype=dtype),
                         weights=torch.rand(INDEX_HEADS, generator=g, device="cuda").to(dtype),
                         index_cache=_randn(g, total, BLOCK, 1, IDX, dtype=dtype), index_block_table=index_table[0],
                         hbm_kpe=hrope.view(-1, BLOCK, KPE), hbm_ckv=hkv.view(-1, BLOCK, CKV),
                         dram_kpe=drope.view(-1, BLOCK, KPE), dram_ckv=dkv.view(-1, BLOCK, CKV),
                         hbm_block_table=table[0], dram_block_table=dram_table[0])}


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind in ("attention", "copy_attention"):
        return _prepare_attention(case, seed)
    if kind in ("indexer_decode", "indexer_prefill"):
        return _prepare_indexer(case, seed)
    if kind == "first_decode":
        return _prepare_first_decode(case, seed)
    return _prepare_step(case, seed)


# ---------------------------------------------------------------------------
# One pass.


def _run_lim(s: dict, query: torch.Tensor) -> None:
    args = (query, s["weights"], s["keys"], s["index_block_table"], s["num_candidate_tokens"], s["num_cache_tokens"],
            s["req_pool_entries"], s["pool"], s["topk_src"], s["topk_dst"])
    if s["case"]["mtp"]:
        ops.fused_li_manage_mtp(*args, s["miss_src"], s["miss_dst"], s["miss_counts"])
    else:
        ops.fused_li_manage(*args, s["miss_counts"])


def _run_step(s: dict) -> dict:
    case = s["case"]
    query = s["queries"][s["turn"]]        # this step's index query
    s["turn"] = (s["turn"] + 1) % len(s["queries"])
    if case["kind"] == "graph":
        l = s["layers"][0]
        out = s["graph"].replay(query_index=query, index_weights=s["weights"], query=l["query"],
                                query_rope=l["query_rope"], index_block_table=s["index_block_table"],
                                hbm_block_table=s["hbm_block_table"], dram_block_table=s["dram_block_table"],
                                num_candidate_tokens=s["num_candidate_tokens"],
                                num_cache_tokens=s["num_cache_tokens"], req_pool_entries=s["req_pool_entries"],
                                actual_seq_lengths_query=s["actual_seq_lengths_query"],
                                actual_seq_lengths_kv=s["actual_seq_lengths_kv"])
        return {**out, "pool": s["pool"], "hbm_kv": l["hbm_kv"], "hbm_rope": l["hbm_rope"]}
    if case["kind"] == "share":
        extra = {"query_index": query, "index_weights": s["weights"]}
        s["stack"].step({f: s[f] for f in CONTEXT_FIELDS}, lambda i: {
            "query_rope": s["layers"][i]["query_rope"], "query": s["layers"][i]["query"], "scale": SCALE,
            "attention_out": s["layers"][i]["out"], **(extra if i == 0 else {})})
        return {**s["stack"].owner_outputs(0, case["batch"]), "pool": s["pool"],
                "layers": [{k: l[k] for k in ("out", "hbm_kv", "hbm_rope")} for l in s["layers"]]}
    _run_lim(s, query)
    got = {k: s[k] for k in ("topk_src", "topk_dst", "miss_counts", "miss_src", "miss_dst", "pool") if k in s}
    if case["kind"] == "lim":
        return got
    l, B = s["layers"][0], case["batch"]
    common = (l["query_rope"], l["query"], s["actual_seq_lengths_query"], s["actual_seq_lengths_kv"],
              s["num_cache_tokens"], s["topk_dst"])
    tables = (s["hbm_block_table"], s["dram_block_table"])
    caches = (l["hbm_rope"], l["hbm_kv"], l["dram_rope"], l["dram_kv"])
    if case["kind"] == "split":
        ops.scatter_copy(s["topk_src"].view(B, TOPK), s["topk_dst"].view(B, TOPK), s["miss_counts"], *tables,
                         caches[0].squeeze(2),
                         caches[1].squeeze(2), *caches[2:])
        ops.sparse_tail_attention(*common, s["hbm_block_table"], l["hbm_rope"], l["hbm_kv"], SCALE, l["out"])
    elif case["mtp"]:
        ops.fused_copy_sfa_mtp(*common, s["topk_src"], s["miss_src"], s["miss_dst"], s["miss_counts"], *tables, *caches,
                               SCALE, l["out"])
    else:
        ops.fused_copy_sfa(*common, s["topk_src"].view(B, TOPK), s["miss_counts"], *tables, *caches, SCALE, l["out"])
    return {**got, "out": l["out"], "hbm_kv": l["hbm_kv"], "hbm_rope": l["hbm_rope"]}


def run(state: dict):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "attention":
        attend = ops.sparse_tail_attention_mtp if case["mtp"] else ops.sparse_tail_attention
        attend(s["query_rope"], s["query"], s["actual_seq_lengths_query"], s["actual_seq_lengths_kv"],
               s["num_cache_tokens"], s["topk_dst"], s["hbm_block_table"], s["hbm_rope"], s["hbm_kv"], SCALE, s["out"])
        return s["out"]
    if kind == "copy_attention":
        ops.fused_copy_sfa(s["query_rope"], s["query"], s["actual_seq_lengths_query"], s["actual_seq_lengths_kv"],
                           s["num_cache_tokens"], s["topk_dst"], s["topk_src"], s["miss_counts"], s["hbm_block_table"],
                           s["dram_block_table"], s["hbm_rope"], s["hbm_kv"], s["dram_rope"], s["dram_kv"], SCALE,
                           s["out"])
        return {"out": s["out"], "hbm_kv": s["hbm_kv"], "hbm_rope": s["hbm_rope"]}
    if kind == "indexer_decode":
        q, w = dsa_indexer_project_query_only(s["hidden"], s["q_c"], s["cos"], s["sin"], s["wq_b"], s["w_proj"], s["q"],
                                              s["w"], n_head=INDEX_HEADS, head_dim=IDX, rope_dim=KPE,
                                              score_scale=IDX ** -0.5)
        return {"q": q, "w": w}
    if kind == "indexer_prefill":
        q, k, w = dsa_indexer_project(s["hidden"], s["q_c"], s["cos"], s["sin"], s["wq_b"], s["wk"], s["k_norm_weight"],
                                      s["k_norm_bias"], s["w_proj"], s["q"], s["k"], s["w"], n_head=INDEX_HEADS,
                                      head_dim=IDX, rope_dim=KPE, score_scale=IDX ** -0.5)
        return {"q": q, "k": k, "w": w}
    if kind == "first_decode":
        ops.initialize_lidu_row(candidate_len=case["prompt"], cache_tokens=case["cache"], cache_slots_row=s["pool"][0],
                                block_size=BLOCK, **s["args"])
        return {"pool": s["pool"], "hbm_kv": s["hbm_kv"], "hbm_rope": s["hbm_rope"]}
    return _run_step(s)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what it has to come to.


def _attention_work(case: dict, c: list[int], kv: list[int], Q: int, distinct: int) -> tuple[float, float]:
    """Bytes and flops of attention over the selected keys and the tails."""
    H, nbytes, flops = case["heads"], 0.0, 0.0
    for budget, length in zip(c, kv):
        tail = length - budget
        nbytes += ROW_BYTES * (tail + (min(budget, distinct) if budget else 0))
        keys = tail + (TOPK if budget else 0)
        flops += 2.0 * Q * H * keys * (CKV + KPE + CKV)
        nbytes += 2.0 * Q * H * (CKV + KPE + CKV)
    return nbytes, flops


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("indexer_decode", "indexer_prefill"):
        T, prefill = case["tokens"], kind == "indexer_prefill"
        nbytes = 2.0 * (T * (HIDDEN + RANK + 2 * KPE) + INDEX_HEADS * IDX * RANK + T * INDEX_HEADS * (IDX + 1))
        nbytes += INDEX_HEADS * HIDDEN * (4.0 if prefill else 2.0)
        flops = 2.0 * T * (INDEX_HEADS * IDX * RANK + INDEX_HEADS * HIDDEN)
        if prefill:
            nbytes += 2.0 * (IDX * HIDDEN + T * IDX)
            flops += 2.0 * T * IDX * HIDDEN
        return {"bytes": nbytes, "flops": flops}
    if kind == "first_decode":
        n, c = case["prompt"], case["cache"]
        return {"bytes": 2.0 * IDX * n + 4.0 * case["width"] + 2.0 * ROW_BYTES * c, "flops": 2.0 * n * INDEX_HEADS * IDX}
    n, c, kv = _lengths(case)
    Q = 4 if case.get("mtp") else 1
    if kind == "attention":
        nbytes, flops = _attention_work(case, c, kv, Q, Q * TOPK)
        return {"bytes": nbytes + 4.0 * TOPK * Q * case["batch"], "flops": flops}
    if kind == "copy_attention":
        nbytes, flops = _attention_work(case, c, kv, 1, TOPK)
        return {"bytes": nbytes + case["batch"] * (8.0 * TOPK + 2.0 * ROW_BYTES * case["misses"]), "flops": flops}
    requests = sum(1 for x in n if x)
    nbytes = 2.0 * IDX * sum(n) + 4.0 * sum(n) + 8.0 * TOPK * Q * requests
    flops = 2.0 * Q * INDEX_HEADS * IDX * sum(n)
    if kind != "lim":
        misses = 0.1 * TOPK * Q * requests     # about a tenth of the selected rows are not cached
        more, macs = _attention_work(case, c, kv, Q, Q * TOPK)
        nbytes += case["layers"] * (more + 2.0 * ROW_BYTES * misses)
        flops += case["layers"] * macs
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    if case["kind"] in ("lim", "first_decode"):
        return "exact"
    # 16-bit results of 32-bit sums: another order of the sums moves a value
    # by one rounding step (2^-8 of a bf16 value) now and then; measured
    # against 64 bits the results are 1.7e-3 off in bf16, 2e-4 in fp16.
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3, "max": 0.04 if case["dtype"] == "bf16" else 5e-3}


def _attend64(query, rope, kv, kr) -> torch.Tensor:
    q = torch.cat((query, rope), -1).double()
    k = torch.cat((kv, kr), -1).double()
    return torch.softmax(SCALE * (q @ k.T.contiguous()), -1) @ kv.double()


def _exact_attention(s: dict) -> torch.Tensor:
    case = s["case"]
    Q = 4 if case.get("mtp") else 1
    kv, rope = s["hbm_kv"].view(-1, CKV), s["hbm_rope"].view(-1, KPE)
    out = torch.zeros(s["out"].shape, dtype=torch.float64, device="cuda")
    lengths, budgets = s["actual_seq_lengths_kv"].tolist(), s["num_cache_tokens"].tolist()
    for r in range(out.shape[0]):
        b = r // Q
        slots = torch.arange(budgets[b], lengths[b] - (Q - 1 - r % Q), device="cuda")
        if budgets[b]:
            slots = torch.cat((s["topk_dst"][r, 0].long(), slots))
        rows = _rows(s["hbm_block_table"][b], slots)
        k, kr = kv[rows], rope[rows]
        if "dram_kv" in s:
            m = s["miss_counts"].tolist()[b]
            src = _rows(s["dram_block_table"][b], s["topk_src"][b, :m])
            k[:m], kr[:m] = s["dram_kv"].view(-1, CKV)[src], s["dram_rope"].view(-1, KPE)[src]
        out[r] = _attend64(s["query"][r], s["query_rope"][r], k, kr)
    return out


def _exact_step(s: dict) -> list[torch.Tensor]:
    """The attention of every layer, from the tokens that 64-bit scores select."""
    case = s["case"]
    Q = 4 if case["mtp"] else 1
    query = s["queries"][0].double()
    n, c, kv = (s[k].tolist() for k in ("num_candidate_tokens", "num_cache_tokens", "actual_seq_lengths_kv"))
    outs = [torch.zeros(l["out"].shape, dtype=torch.float64, device="cuda") for l in s["layers"]]
    for r in range(s["rows"]):
        b = r // Q
        tail = torch.arange(c[b], kv[b] - (Q - 1 - r % Q), device="cuda")
        src = torch.empty(0, dtype=torch.int64, device="cuda")
        if c[b]:
            keys = s["keys"].view(-1, IDX)[_rows(s["index_block_table"][b], torch.arange(n[b], device="cuda"))].double()
            src = _rows(s["dram_block_table"][b], torch.topk(_scores(keys, query[r], s["weights"][r].double()), TOPK).indices)
        dst = _rows(s["hbm_block_table"][b], tail)
        for l, out in zip(s["layers"], outs):
            out[r] = _attend64(l["query"][r], l["query_rope"][r],
                               torch.cat((l["dram_kv"].view(-1, CKV)[src], l["hbm_kv"].view(-1, CKV)[dst])),
                               torch.cat((l["dram_rope"].view(-1, KPE)[src], l["hbm_rope"].view(-1, KPE)[dst])))
    return outs


def _rope64(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    x = x.clone()
    e, o = x[..., 0:KPE:2].clone(), x[..., 1:KPE:2].clone()
    x[..., 0:KPE:2] = e * cos[..., 0::2] - o * sin[..., 0::2]
    x[..., 1:KPE:2] = o * cos[..., 1::2] + e * sin[..., 1::2]
    return x


def _exact_indexer(s: dict) -> dict:
    T = s["q"].shape[0]
    cos, sin, hidden = s["cos"].double(), s["sin"].double(), s["hidden"].double()
    q = (s["q_c"].double() @ s["wq_b"].double().T).view(T, INDEX_HEADS, IDX)
    got = {"q": _rope64(q, cos[:, None], sin[:, None]), "w": hidden @ s["w_proj"].double().T * IDX ** -0.5}
    if "wk" in s:
        k = torch.nn.functional.layer_norm(hidden @ s["wk"].double().T, (IDX,), s["k_norm_weight"].double(),
                                           s["k_norm_bias"].double(), 1e-6)
        got["k"] = _rope64(k, cos, sin)
    return got


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("lim", "first_decode"):
        return None                            # whole numbers and copied rows
    s = prepare(case, seed)
    if kind.startswith("indexer"):
        return _exact_indexer(s)
    if kind == "attention":
        return _exact_attention(s)
    if kind == "copy_attention":
        return {"out": _exact_attention(s), "hbm_kv": None, "hbm_rope": None}
    outs = _exact_step(s)
    if kind == "share":
        return {"layers": [{"out": o, "hbm_kv": None, "hbm_rope": None} for o in outs]}
    return {"attention_out" if kind == "graph" else "out": outs[0]}
