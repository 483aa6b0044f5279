"""Timed cases of the retrieval path: what programs built on retrieve_amd have it do.

Each case is one call (or the one fixed pair of calls) that such a program makes again and again:
a LiNR or SilverTorch module's forward over a query batch, a fused scan over a large table, or one
index build. Sizes are the repository's own workloads (``bench.py``: 30M x 512 int8, 10M x 128
bf16, 30M 512-bit codes, 100k x 128 fp32) and catalogue sizes between them, with batches from one
query to 1024. Items, attributes and queries come from the seed alone; everything is on the GPU.

``FAMILIES`` names the kinds of call; ``listed`` holds twelve of them at set sizes, ``draw`` picks
a kind and sizes of the same ranges.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import retrieve_amd.hip  # noqa: F401  (registers torch.ops.retrieve.* / retrieve_amd.*)
import retrieve_amd.st as st
from retrieve_amd import bloom as bl
from retrieve_amd import modules as mods

DEV = "cuda:0"
# attribute cardinalities: the module cases' four, the filtered full scans' eight (bench.py's)
CARDS4 = (16, 64, 256, 1000)
CARDS8 = (16, 32, 64, 128, 256, 512, 1000, 1000)
BLOOM_BITS, BLOOM_K, HASH_K = 64, 3, 7  # Bloom bits an item, hash positions a token, stored hashes
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


# --- the cases --------------------------------------------------------------------------------


def listed():
    return [
        # the smallest call: one user's request over a small catalogue, where latency counts
        {"name": "v1_fp16_100k_b1", "family": "v1", "n": 100_000, "d": 128, "b": 1, "k": 100,
         "filtered": False},
        # a serving batch over a mid-size catalogue, the attribute filter folded into the scan
        {"name": "v1_exact_800k_b16", "family": "v1", "n": 800_003, "d": 128, "b": 16, "k": 100,
         "filtered": True},
        # the pre-filter form: passing ids compacted, then re-scored exactly
        {"name": "v2_exact_800k_b16", "family": "v2", "n": 800_003, "d": 128, "b": 16, "k": 100},
        # the default 1-bit shortlist (pool 5000) under a filter, then the exact re-score
        {"name": "v3_exact_3m_b16", "family": "v3", "n": 3_000_000, "d": 128, "b": 16, "k": 100,
         "pool": 5000, "filtered": True},
        # IVF + int8 under the exact filter, int32 keys: a batch of 64
        {"name": "ivf_exact_3m_b64", "family": "ivf", "n": 3_000_000, "d": 128, "b": 64, "k": 100,
         "lists": 1024, "probes": 64, "mode": "exact", "path": "int32"},
        # IVF + int8 with Bloom plans and their recheck, fp16 keys (the serving defaults)
        {"name": "ivf_bloom_10m_b16", "family": "ivf", "n": 10_000_000, "d": 256, "b": 16,
         "k": 100, "lists": 4096, "probes": 128, "mode": "bloom", "path": "fp16"},
        # the headline workload of bench.py: filtered int8 top-100 over 30M x 512
        {"name": "int8_bloom_30m_b16", "family": "int8", "n": 30_000_000, "d": 512, "b": 16,
         "k": 100, "filtered": True},
        # exact fp32 retrieval of a large evaluation batch over a small table (bench.py exact)
        {"name": "knn_fp32_100k_b1024", "family": "knn", "dtype": "fp32", "n": 100_000, "d": 128,
         "b": 1024, "k": 100},
        # a wide embedding at a ragged batch
        {"name": "knn_fp16_1m_d384_b50", "family": "knn", "dtype": "fp16", "n": 1_000_000,
         "d": 384, "b": 50, "k": 100},
        # offline retrieval over the large bf16 table (bench.py dense): the largest case
        {"name": "knn_bf16_10m_b1024", "family": "knn", "dtype": "bf16", "n": 10_000_000,
         "d": 128, "b": 1024, "k": 100},
        # two-stage 1-bit retrieval: filtered Hamming top-1000, int8 re-rank (bench.py binary)
        {"name": "bits_rerank_30m_b256", "family": "bits", "n": 30_000_000, "bits": 512,
         "b": 256, "k": 100, "pool": 1000},
        # building the codes of an index: int8 per row and global, 1-bit codes, the Bloom words
        {"name": "build_3m_d128", "family": "build", "n": 3_000_000, "d": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["v1", "v1", "v2", "v3", "ivf", "ivf", "int8", "knn", "knn", "bits",
                         "build"])
    k = _log_int(rng, 10, 1000)
    b = _log_int(rng, 1, 256)
    if family in ("v1", "v2"):
        # (v2 writes the passing ids of every query: batches of one to 64)
        c = {"n": _log_int(rng, 50_000, 2_000_000 if family == "v2" else 5_000_000),
             "d": rng.choice([32, 64, 128, 256, 384, 512]),
             "b": min(b, 64) if family == "v2" else b, "k": k}
        if family == "v1":
            c["filtered"] = rng.random() < 0.6
    elif family == "v3":
        pool = rng.choice([200, 800, 2000, 5000, 8000])
        c = {"n": _log_int(rng, 100_000, 6_000_000), "d": rng.choice([64, 128, 256]),
             "b": min(b, 64), "k": min(k, pool), "pool": pool, "filtered": rng.random() < 0.6}
    elif family == "ivf":
        lists = rng.choice([256, 1000, 1024, 4096])
        c = {"n": _log_int(rng, 300_000, 10_000_000), "d": rng.choice([64, 128, 192, 256, 512]),
             "b": min(b, 128), "k": k, "lists": lists,
             "probes": _log_int(rng, 8, lists // 8),
             "mode": rng.choice(["none", "exact", "bloom"]), "path": rng.choice(["int32", "fp16"])}
    elif family == "int8":
        filtered = rng.random() < 0.5
        c = {"n": _log_int(rng, 100_000, 30_000_000),
             "d": 512 if filtered else rng.choice([64, 128, 256, 512, 768, 1024]),
             "b": b, "k": k, "filtered": filtered}
        c["n"] = min(c["n"], 30_000_000 * 512 // max(512, c["d"]))
    elif family == "knn":
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        d = rng.choice([32, 64, 128] if dtype == "fp32" else [32, 64, 128, 256, 384, 512])
        c = {"dtype": dtype, "n": _log_int(rng, 20_000, 400_000 if dtype == "fp32" else 5_000_000),
             "d": d, "b": _log_int(rng, 1, 1024), "k": k}
    elif family == "bits":
        c = {"n": _log_int(rng, 300_000, 30_000_000), "bits": 512, "b": max(8, b),
             "k": min(k, 200), "pool": rng.choice([200, 500, 1000])}
    else:
        d = rng.choice([64, 128, 192, 256, 512])
        c = {"n": _log_int(rng, 100_000, 3_000_000 * 128 // max(128, d)), "d": d}
    c["n"] |= 1  # odd row counts
    return {"family": family, **c}


# --- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _unit(n, d, g, dtype=torch.float32, chunk=1 << 20):
    """N(0, 1) rows, L2-normalised in fp32."""
    out = torch.empty((n, d), dtype=dtype, device=DEV)
    for s in range(0, n, chunk):
        m = min(chunk, n - s)
        out[s:s + m] = torch.nn.functional.normalize(
            torch.randn((m, d), generator=g, device=DEV), dim=1)
    return out


def _int8(n, d, g, chunk=1 << 21):
    """int8 codes of N(0, 1) rows, their largest value near three and a half sigma."""
    out = torch.empty((n, d), dtype=torch.int8, device=DEV)
    for s in range(0, n, chunk):
        m = min(chunk, n - s)
        out[s:s + m] = torch.randn((m, d), generator=g, device=DEV).mul_(36.0).round_() \
            .clamp_(-127, 127)
    return out


def _words(n, w, g, chunk=1 << 22):
    """Random 64-bit code words: the sign bits of a Gaussian projection of Gaussian rows."""
    out = torch.empty((n, w), dtype=torch.int64, device=DEV)
    for s in range(0, n, chunk):
        m = min(chunk, n - s)
        out[s:s + m] = torch.randint(-(2**63), 2**63 - 1, (m, w), generator=g, device=DEV)
    return out


def _zipf(card):
    p = 1.0 / np.arange(1, card + 1, dtype=np.float64) ** 1.1
    return p / p.sum()


def _attrs(n, cards, g, dtype):
    """[N, C, 1] attribute values, Zipf(1.1) over each attribute's cardinality."""
    out = torch.empty((n, len(cards), 1), dtype=dtype, device=DEV)
    for c, card in enumerate(cards):
        cdf = torch.from_numpy(np.cumsum(_zipf(card))).float().to(DEV)
        out[:, c, 0] = torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV)) \
            .clamp_(max=card - 1)
    return out


def _query_values(b, seed):
    """[B, 4] single-value clauses: one or two active attributes, frequent values, so that a
    query passes about 2 to 25 % of the items."""
    r = np.random.default_rng(seed)
    q = np.full((b, len(CARDS4)), -1, np.int64)
    for row in range(b):
        if row % 2 == 0:
            q[row, r.integers(0, 4)] = r.integers(0, 3)
        else:
            for c in r.choice(4, 2, replace=False):
                q[row, c] = r.integers(0, 2)
    return torch.from_numpy(q).to(DEV)


def _query_sets(b, seed, selectivity=0.1):
    """[B, 8, V] value sets: an AND over one to three attributes of an OR over their most
    frequent values, about ``selectivity`` of the items passing (bench.py's query sets)."""
    r = np.random.default_rng(seed)
    rows = []
    for row in range(b):
        picked = r.choice(len(CARDS8), 1 + row % 3, replace=False)
        target = selectivity ** (1.0 / len(picked))
        sets = [[] for _ in CARDS8]
        for c in picked:
            p, mass, v = _zipf(CARDS8[c]), 0.0, int(r.integers(0, 2))
            while mass < target and v < CARDS8[c]:
                sets[c].append(v)
                mass += p[v]
                v += 1
        rows.append(sets)
    width = max(len(s) for sets in rows for s in sets)
    out = np.full((b, len(CARDS8), width), -1, np.int64)
    for i, sets in enumerate(rows):
        for c, s in enumerate(sets):
            out[i, c, :len(s)] = s
    return out


class _Filter:
    """The filtered full scans' attributes, Bloom index and query plans (bench.py's)."""

    def __init__(self, n, b, g, seed):
        self.attrs = _attrs(n, CARDS8, g, torch.int16)
        sets = _query_sets(b, seed)
        self.words, self.offs = torch.ops.st.bloom_index_build_fixed(
            *st.attrs_to_features(self.attrs.long()), BLOOM_BITS, BLOOM_K)
        self.doc_bits = torch.ops.retrieve_amd.bloom_doc_bits(self.words, self.offs, n)
        self.blob, self.plans, self.stack = st.prepare_plans(
            bl.sets_to_expressions(sets), HASH_K, torch.device(DEV))
        self.rev = torch.zeros(len(CARDS8), dtype=torch.bool, device=DEV)
        self.sets = torch.from_numpy(sets).to(DEV)


def _ivf_parts(case, seed):
    """An IVF index as a state dict (a build's result, loaded): centroids, cluster-sorted codes
    of rows around them under one global scale, the layout, and the filter's tables."""
    g = _gen(seed)
    n, d, lists = case["n"], case["d"], case["lists"]
    cent = torch.randn((lists, d), generator=g, device=DEV)
    # cluster masses spread over about a factor of four, as k-means leaves them
    mass = torch.rand(lists, generator=g, device=DEV) + 0.3
    cdf = torch.cumsum(mass, 0) / mass.sum()
    u = torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV)).clamp_(max=lists - 1)
    perm = torch.argsort(u, stable=True)
    us = u[perm]
    codes = torch.empty((n, d), dtype=torch.int8, device=DEV)
    scale = 5.5 / 127.0
    for s in range(0, n, 1 << 20):
        x = cent[us[s:s + (1 << 20)]] + 0.7 * torch.randn(
            (min(1 << 20, n - s), d), generator=g, device=DEV)
        codes[s:s + (1 << 20)] = (x / scale).round_().clamp_(-127, 127)
    sizes = torch.bincount(u, minlength=lists)
    offsets = torch.zeros(lists + 1, dtype=torch.int64, device=DEV)
    offsets[1:] = sizes.cumsum(0)
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(n, device=DEV)
    parts = {"centroids": cent, "item_codes": codes, "cluster_offsets": offsets,
             "cluster_sizes": sizes, "sort_perm": perm, "inv_perm": inv,
             "global_scale": torch.tensor(scale, device=DEV)}
    at = torch.randint(0, lists, (case["b"],), generator=g, device=DEV)
    query = cent[at] + 0.7 * torch.randn((case["b"], d), generator=g, device=DEV)
    attrs = _attrs(n, CARDS4, g, torch.int64) if case["mode"] != "none" else None
    return parts, query, attrs


def _ivf_state(case, seed):
    parts, query, attrs = _ivf_parts(case, seed)
    prepared = None
    if attrs is not None:
        slots, clause_slots = mods.fork_clause_attrs(attrs)  # rows already in sorted order
        parts.update(item_clause_attrs=slots, clause_slots=clause_slots,
                     clause_is_reverse=torch.zeros(len(CARDS4), dtype=torch.bool, device=DEV))
    bloom = case["mode"] == "bloom"
    if bloom:
        parts["bloom_index"], parts["bundle_b_offsets"] = torch.ops.st.bloom_index_build_fixed(
            *st.attrs_to_features(attrs), BLOOM_BITS, BLOOM_K)
    module = mods.SilverTorch(
        case["k"], case["lists"], case["probes"], filter_mode=case["mode"],
        m_bits=BLOOM_BITS if bloom else None, k_hash=BLOOM_K if bloom else None,
        official=mods.OfficialConfig(score_path=case["path"]))
    mods.load_prebuilt(module, parts)
    if attrs is not None:
        prepared = module.prepare_queries(_query_values(case["b"], seed))
    return {"module": module, "query": query, "prepared": prepared}


def _linr_inputs(case, seed):
    g = _gen(seed)
    items = _unit(case["n"], case["d"], g)
    query = _unit(case["b"], case["d"], g)
    attrs = values = None
    if case["family"] == "v2" or case["filtered"]:
        attrs = _attrs(case["n"], CARDS4, g, torch.int64)
        values = _query_values(case["b"], seed)
    return items, query, attrs, values


def _knn_inputs(case, seed):
    g = _gen(seed)
    dtype = DTYPES[case["dtype"]]
    return _unit(case["n"], case["d"], g, dtype), _unit(case["b"], case["d"], g, dtype)


def _build_inputs(case, seed):
    g = _gen(seed)
    embs = torch.randn((case["n"], case["d"]), generator=g, device=DEV)
    return embs, torch.randperm(case["n"], generator=g, device=DEV), \
        _attrs(case["n"], CARDS4, g, torch.int64)


def prepare(case, seed):
    family = case["family"]
    state = {"family": family, "case": dict(case)}
    if family in ("v1", "v2", "v3"):
        items, query, attrs, values = _linr_inputs(case, seed)
        flt = None if attrs is None else mods.ExactAttributeFilter()
        if family == "v1":
            module = mods.LiNRV1(case["k"], filter=flt)
        elif family == "v2":
            module = mods.LiNRV2(case["k"], filter=flt)
        else:
            module = mods.LiNRV3(case["k"], candidate_pool=case["pool"], filter=flt)
        module.register_index(items, attrs)
        state.update(module=module, query=query,
                     prepared=None if flt is None else module.prepare_queries(values))
    elif family == "ivf":
        state.update(_ivf_state(case, seed))
    elif family == "int8":
        g = _gen(seed)
        state.update(items=_int8(case["n"], case["d"], g), query=_int8(case["b"], case["d"], g),
                     flt=_Filter(case["n"], case["b"], g, seed) if case["filtered"] else None)
    elif family == "knn":
        items, query = _knn_inputs(case, seed)
        module = mods.FullScanKNN(case["k"])
        module.register_index(items)
        state.update(module=module, query=query)
    elif family == "bits":
        g = _gen(seed)
        n, b = case["n"], case["b"]
        state.update(item_bits=_words(n, case["bits"] // 64, g),
                     query_bits=_words(b, case["bits"] // 64, g), item_codes=_int8(n, 512, g),
                     query_codes=_int8(b, 512, g), flt=_Filter(n, b, g, seed),
                     counts=torch.full((b,), case["pool"], dtype=torch.int64, device=DEV))
    else:
        embs, perm, attrs = _build_inputs(case, seed)
        state.update(embs=embs, perm=perm, features=st.attrs_to_features(attrs))
    return state


# --- one pass ---------------------------------------------------------------------------------


def run(state):
    case, family = state["case"], state["family"]
    ops = torch.ops.retrieve_amd
    if family in ("v1", "v2", "v3", "ivf"):
        if state["prepared"] is None:
            return state["module"](state["query"])
        return state["module"](state["query"], state["prepared"])
    if family == "knn":
        return state["module"](state["query"])
    flt = state.get("flt")
    if family == "int8":
        if flt is None:
            return ops.int8_scan_topk(state["query"], state["items"], case["k"])
        return ops.scan_topk_bloom_clauses(
            state["query"], state["items"], case["k"], flt.attrs, flt.rev, flt.sets, flt.doc_bits,
            flt.words, flt.offs, flt.blob, flt.plans, flt.stack, BLOOM_K, HASH_K)
    if family == "bits":
        words = st.bloom_search_t(flt.words, flt.offs, flt.blob, flt.plans, flt.stack, BLOOM_K,
                                  HASH_K)
        ids, scores = ops.hamming_scan_topk_clauses(
            state["query_bits"], state["item_bits"], case["pool"], flt.attrs, flt.rev, flt.sets,
            words)
        return ids, scores, ops.int8_candidates_topk(
            state["query_codes"], state["item_codes"], ids, state["counts"], case["k"])
    embs = state["embs"]
    row_codes, row_scales = ops.quantize_int8(embs)
    codes, scale = mods.quantize_int8_global(embs, rows=state["perm"])
    onebit = mods.OneBitKNN(1)
    onebit.register_index(embs)
    index, offsets = torch.ops.st.bloom_index_build_fixed(*state["features"], BLOOM_BITS, BLOOM_K)
    return row_codes, row_scales, codes, scale, onebit.item_bits, index, offsets


# --- what a pass cannot do without ------------------------------------------------------------


def work(case):
    family, n, b, k = case["family"], case["n"], case.get("b", 0), case.get("k", 0)
    d = case.get("d", 0)
    out = b * k * 12  # ids and scores
    if family == "build":
        # rows and attributes read once; two int8 tables, scales, codes and Bloom words written
        return {"bytes": n * (d * 4 + len(CARDS4) * 8 + 8) + n * (2 * d + 4 + d // 8 + 8),
                "flops": n * d * 8}
    if family == "bits":
        # codes and Bloom words once, the re-ranked rows once a query
        return {"bytes": n * (case["bits"] // 8 + 8) + b * case["pool"] * 512 + out,
                "flops": 2 * b * n * case["bits"] // 4}  # a 1-bit product counted as a quarter
    if family == "int8":
        return {"bytes": n * d + b * d + out, "flops": b * n * d}  # an int8 product as half
    if family == "ivf":
        share = case["probes"] / case["lists"]
        rows = n * (1 - (1 - share) ** b)  # rows that some query probes
        attr = 0 if case["mode"] == "none" else rows * len(CARDS4) * 4
        return {"bytes": rows * d + attr + out + case["lists"] * d * 4,
                "flops": b * n * share * d + 2 * b * case["lists"] * d}
    esize = 4 if case.get("dtype") == "fp32" else 2
    attr = n * len(CARDS4) * 8 if family == "v2" or case.get("filtered") else 0
    if family == "v2":
        rows = n * (1 - 0.9 ** b)
        return {"bytes": attr + rows * d * 2 + b * d * 4 + out, "flops": 2 * b * 0.1 * n * d}
    if family == "v3":
        return {"bytes": attr + n * d // 8 + b * case["pool"] * d * 2 + out,
                "flops": 2 * b * n * d // 4 + 2 * b * case["pool"] * d}
    return {"bytes": attr + n * d * esize + b * d * esize + out, "flops": 2 * b * n * d}


# --- tolerances and 64-bit results --------------------------------------------------------------


def tolerance(case):
    family = case["family"]
    if family in ("int8", "bits", "build"):
        return "exact"  # integer dots and codes, one fixed fp32 division a scale
    if family == "ivf":
        # integer dots; the probed lists come from fp32 centroid products, which round by order
        return {"rel": 1e-6, "max": 1e-2, "differ": 0.005}
    if case.get("dtype") in ("bf16", "fp16"):
        # fp32 sums rounded once to 16 bits, whose ties follow the sums' last bits
        # (one last place: 2^-10 of a value in fp16, 2^-7 in bf16; few values sit on such a tie)
        return {"rel": 3e-5 if case["dtype"] == "fp16" else 2e-4,
                "max": 1e-3 if case["dtype"] == "fp16" else 8e-3, "differ": 0.01}
    # fp32 sums: ids change places where scores agree to their last bits
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}


def _pass_rows(attrs, values):
    """[B, N] bool: every active clause's value is the item's."""
    ok = torch.ones((values.shape[0], attrs.shape[0]), dtype=torch.bool, device=DEV)
    for c in range(attrs.shape[1]):
        v = values[:, c:c + 1]
        ok &= (attrs[:, c, 0][None] == v) | (v == -1)
    return ok


def _topk64(query, items, k, ok=None, chunk=1 << 18):
    """The k best 64-bit products of every query over the items that pass, best first."""
    q = query.double()
    best = torch.full((q.shape[0], k), -math.inf, dtype=torch.float64, device=DEV)
    for s in range(0, items.shape[0], chunk):
        sc = q @ items[s:s + chunk].double().t()
        if ok is not None:
            sc.masked_fill_(~ok[:, s:s + chunk], -math.inf)
        best = torch.topk(torch.cat([best, sc], 1), k, dim=1).values
    return best


def exact(case, seed):
    family, k = case["family"], case.get("k", 0)
    if family in ("int8", "bits"):
        return None  # whole numbers, which the comparison wants equal
    if family == "build":
        embs, _, _ = _build_inputs(case, seed)
        a = torch.cat([x.double().abs().amax(1) for x in embs.split(1 << 20)]).clamp_min(1e-8)
        return None, a / 127.0, None, float(a.max() / 127.0), None, None, None
    if family == "knn":
        items, query = _knn_inputs(case, seed)
        return None, _topk64(query, items, k)
    if family == "ivf":
        parts, query, attrs = _ivf_parts(case, seed)
        a = query.abs().amax(1, keepdim=True).clamp_min(1e-8).double()
        codes = (query.double() / a * 127.0).round().clamp(-128, 127)
        probed = torch.zeros((case["b"], case["lists"]), dtype=torch.bool, device=DEV)
        top = torch.topk(query.double() @ parts["centroids"].double().t(), case["probes"], dim=1)
        probed.scatter_(1, top.indices, True)
        of = torch.repeat_interleave(torch.arange(case["lists"], device=DEV),
                                     parts["cluster_sizes"])
        ok = probed[:, of]
        if attrs is not None:
            ok &= _pass_rows(attrs, _query_values(case["b"], seed))
        dots = _topk64(codes, parts["item_codes"], k, ok)
        return None, dots * (a / 127.0) * parts["global_scale"].double()
    items, query, attrs, values = _linr_inputs(case, seed)
    ok = None if attrs is None else _pass_rows(attrs, values)
    half_i, half_q = items.half(), query.half()
    if family == "v3":
        # the codes are the rows' signs in some fixed order: the Hamming order is that of the
        # sign products, ties to the lower id
        n = items.shape[0]
        keys = torch.empty((case["b"], n), dtype=torch.float64, device=DEV)
        sq = torch.where(query > 0, 1.0, -1.0)
        for s in range(0, n, 1 << 20):
            keys[:, s:s + (1 << 20)] = sq @ torch.where(items[s:s + (1 << 20)] > 0, 1.0, -1.0).t()
        keys = keys * n - torch.arange(n, device=DEV, dtype=torch.float64)
        if ok is not None:
            keys.masked_fill_(~ok, -math.inf)
        pool = torch.topk(keys, case["pool"], dim=1)
        rows = half_i[pool.indices].double()  # [B, pool, D]
        sc = (rows * half_q.double()[:, None]).sum(-1)
        sc.masked_fill_(pool.values == -math.inf, -math.inf)
        return None, torch.topk(sc, k, dim=1).values
    return None, _topk64(half_q, half_i, k, ok)
