"""Workloads whose speed this repository is judged by, through its public entry points.

A case is a dict of plain values; ``kind`` names the entry point:

  step       CompressionPipeline.step: phases, scores, statistics, aggregate,
             selection, compaction and block-table rewrite of a batch
  compress   TriAttentionMethod.compress_batch, the method API a serving
             worker calls when requests cross their KV budget
  score      CompressionPipeline.score + aggregate: the scoring stage alone
  layer      kernels.score_paged_keys_mean_precomputed: one layer's scores
  select     selection.select_keep_indices_batched on given scores
  compact    CompressionPipeline.compact with a given keep set
  calibrate  calibration.LayerAccumulator over hooked query projections

Sequence lengths are spread evenly at random over [min_len, max_len] (the same
for every seed of a case).  Keys and values are normal with a per-channel
scale, calibration centres are random complex vectors.
"""

from __future__ import annotations

import math
import os
import random
import sys
import tempfile
from pathlib import Path
from types import SimpleNamespace

import torch

_ROOT = Path(__file__).resolve().parents[1] / "vllm-ascend-kvcompress-hust_amd"
if str(_ROOT) not in sys.path:
    sys.path.insert(0, str(_ROOT))

from kvcompress_mi355x import calibration  # noqa: E402
from kvcompress_mi355x.methods import create_method  # noqa: E402
from kvcompress_mi355x.methods.base import CompressionRequest, LayerCache, ModelShape  # noqa: E402
from kvcompress_mi355x.methods.triattention import kernels, selection  # noqa: E402
from kvcompress_mi355x.methods.triattention.method import COMPACTION_ORDER_ENV  # noqa: E402
from kvcompress_mi355x.methods.triattention.pipeline import Batch, CompressionPipeline, ScoringTables  # noqa: E402
from kvcompress_mi355x.methods.triattention.scoring import build_geometric_offsets  # noqa: E402
from kvcompress_mi355x.methods.triattention.stats import DeviceLayerCalibrationStats  # noqa: E402

PAGE = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Attention shapes of the repository's workloads, and generic ones: query
# heads, KV heads, head dim, rotated dims, RoPE base.
_QWEN25 = {"heads": 40, "kv": 8, "head_dim": 128, "rotary": 128, "theta": 1e6}
_QWEN35 = {"heads": 16, "kv": 2, "head_dim": 256, "rotary": 64, "theta": 1e7}
_GLOBAL = {"policy": "global", "segments": 8, "prefix": 0}


def listed():
    return [
        # The smallest call: one layer, one 4096-token sequence (launches and
        # latency count), as the tiny correctness workload.
        {"name": "step-1x4096", "kind": "step", "heads": 8, "kv": 2, "head_dim": 128, "rotary": 128, "theta": 1e6,
         "dtype": "bf16", "style": "half", "aggregation": "mean", "layers": 1, "stride": 1, "n_seq": 1,
         "min_len": 4096, "max_len": 4096, "budget": 2048, "recent": 128, "max_model_len": 32768, **_GLOBAL},
        # The everyday call of a server: one request has just crossed its
        # budget and is compressed in all 48 layers.
        {"name": "compress-1x4600", "kind": "compress", **_QWEN25, "dtype": "bf16", "style": "half",
         "aggregation": "mean", "layers": 48, "stride": 8, "n_seq": 1, "min_len": 4600, "max_len": 4600,
         "budget": 4096, "recent": 128, "max_model_len": 32768, **_GLOBAL},
        # Several requests of one scheduler output, fp16, ragged.
        {"name": "compress-6x4k-9k-fp16", "kind": "compress", **_QWEN25, "dtype": "fp16", "style": "half",
         "aggregation": "mean", "layers": 24, "stride": 8, "n_seq": 6, "min_len": 4224, "max_len": 9000,
         "budget": 4096, "recent": 128, "max_model_len": 32768, **_GLOBAL},
        # The scoring stage of the headline batch (6 scoring layers).
        {"name": "score-16x16384", "kind": "score", **_QWEN25, "dtype": "bf16", "style": "half",
         "aggregation": "mean", "layers": 6, "n_seq": 16, "min_len": 16384, "max_len": 16384, "max_model_len": 32768},
        # Hybrid model: partial RoPE, head_dim 256, ragged long sequences.
        {"name": "score-hybrid-8x8k-64k", "kind": "score", **_QWEN35, "dtype": "bf16", "style": "half",
         "aggregation": "mean", "layers": 5, "n_seq": 8, "min_len": 8192, "max_len": 65536, "max_model_len": 262144},
        # score_aggregation "max" on the headline shape.
        {"name": "score-max-8x16384", "kind": "score", **_QWEN25, "dtype": "bf16", "style": "half",
         "aggregation": "max", "layers": 6, "n_seq": 8, "min_len": 16384, "max_len": 16384, "max_model_len": 32768},
        # Head sizes between the powers of two are ordinary too: head_dim 96.
        {"name": "score-hd96-8x2k-16k", "kind": "score", "heads": 32, "kv": 8, "head_dim": 96, "rotary": 96,
         "theta": 1e4, "dtype": "bf16", "style": "half", "aggregation": "mean", "layers": 4, "n_seq": 8,
         "min_len": 2048, "max_len": 16384, "max_model_len": 32768},
        # One layer of one tensor-parallel rank's share of the hybrid model, the
        # call the reference publishes a speed-up for.
        {"name": "layer-1kv-32768", "kind": "layer", "heads": 8, "kv": 1, "head_dim": 256, "rotary": 64, "theta": 1e7,
         "dtype": "bf16", "style": "half", "aggregation": "mean", "layers": 1, "n_seq": 1, "min_len": 32768,
         "max_len": 32768, "max_model_len": 262144},
        # Keep-set selection of a few very long sequences.
        {"name": "select-4x131072", "kind": "select", "n_seq": 4, "min_len": 131072, "max_len": 131072,
         "budget": 4608, "recent": 256, **_GLOBAL},
        # Compaction of the headline batch into private pages (a third of its layers).
        {"name": "compact-16x4096", "kind": "compact", **_QWEN25, "dtype": "bf16", "layers": 16, "n_seq": 16,
         "min_len": 16384, "max_len": 16384, "budget": 4096, "recent": 128, "inplace": False},
        # Compaction in place when the pool has no free page.
        {"name": "compact-inplace-4x4608", "kind": "compact", **_QWEN25, "dtype": "bf16", "layers": 8, "n_seq": 4,
         "min_len": 65536, "max_len": 131072, "budget": 4608, "recent": 256, "inplace": True},
        # Calibration statistics of a 4096-token pass over hooked projections.
        {"name": "calibrate-8x4096", "kind": "calibrate", "heads": 40, "head_dim": 128, "rotary": 128,
         "dtype": "bf16", "layers": 8, "tokens": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Head shapes a drawn case takes: (head_dim, rotated dims).
_SHAPES = ((64, 64), (80, 80), (96, 96), (128, 128), (128, 64), (128, 32), (192, 192), (256, 64), (256, 256))


def draw(rng):
    kind = rng.choice(("step", "compress", "score", "score", "score", "layer", "select", "compact", "calibrate"))
    if kind == "calibrate":
        head_dim, rotary = rng.choice(_SHAPES)
        return {"kind": kind, "heads": rng.randint(4, 40), "head_dim": head_dim, "rotary": rotary,
                "dtype": rng.choice(("bf16", "fp16", "fp32")), "layers": rng.randint(1, 6), "tokens": _log_int(rng, 64, 4096)}
    if kind == "select":
        n_seq = _log_int(rng, 1, 64)
        hi = _log_int(rng, 1024, min(262144, (1 << 20) // n_seq))
        lo = max(513, _log_int(rng, max(513, hi // 8), hi))
        budget = rng.randint(256, min(lo, 4608))
        return {"kind": kind, "n_seq": n_seq, "min_len": min(lo, hi), "max_len": hi, "budget": budget,
                "recent": rng.randint(0, min(256, budget // 2)), "policy": rng.choice(("global", "v3")),
                "segments": rng.randint(2, 12), "prefix": rng.choice((0, 4, 64))}
    head_dim, rotary = rng.choice(_SHAPES)
    kv = rng.choice((1, 2, 4, 8))
    qpk = rng.randint(1, 8)
    row = kv * head_dim * 2
    shape = {"heads": kv * qpk, "kv": kv, "head_dim": head_dim, "rotary": rotary, "theta": rng.choice((1e4, 1e6, 1e7)),
             "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    if kind == "layer":
        n = _log_int(rng, 300, 65536)
        return {"kind": kind, **shape, "style": rng.choice(("half", "half", "interleaved")), "aggregation": "mean", "layers": 1,
                "n_seq": 1, "min_len": n, "max_len": n, "max_model_len": 131072}
    if kind == "score":
        layers, n_seq = rng.randint(1, 6), _log_int(rng, 1, 48)
        aggregation = rng.choice(("mean", "mean", "max"))
        # Bytes of keys at most about those of the headline batch (a fifth for "max").
        cap = (3e9 if aggregation == "mean" else 6e8) / (layers * n_seq * row)
        hi = _log_int(rng, 600, max(700, min(131072, int(cap))))
        lo = _log_int(rng, max(300, hi // 6), hi)
        return {"kind": kind, **shape, "style": rng.choice(("half", "half", "interleaved")), "aggregation": aggregation,
                "layers": layers, "n_seq": n_seq, "min_len": lo, "max_len": hi, "max_model_len": rng.choice((32768, 131072))}
    if kind == "compact":
        layers, n_seq = rng.randint(2, 24), _log_int(rng, 1, 48)
        budget = _log_int(rng, 300, max(320, min(4608, int(5e9 / (layers * n_seq * row * 4)))))
        hi = budget + _log_int(rng, 100, max(120, min(60000, int(1.5e10 / (layers * n_seq * row * 2)))))
        lo = rng.randint(budget + 64, hi)
        return {"kind": kind, **shape, "layers": layers, "n_seq": n_seq, "min_len": lo, "max_len": hi, "budget": budget,
                "recent": rng.randint(0, min(256, budget // 2)), "inplace": rng.choice((False, False, True))}
    # step, compress: a few sequences, every layer compacted.
    layers, n_seq = _log_int(rng, 1, 32), _log_int(rng, 1, 4)
    budget = _log_int(rng, 512, max(520, min(4608, int(3e9 / (layers * n_seq * row * 4))))) // PAGE * PAGE
    hi = budget + 200 + _log_int(rng, 64, 8192)
    lo = rng.randint(budget + 150, hi)
    extra = {"policy": rng.choice(("global", "v3")), "segments": rng.randint(2, 10), "prefix": rng.choice((0, 4, 64))}
    return {"kind": kind, **shape, "style": "half", "aggregation": "mean", "layers": layers,
            "stride": rng.randint(1, max(1, min(8, layers))), "n_seq": n_seq, "min_len": lo, "max_len": hi, "budget": budget,
            "recent": rng.randint(1, 128), "max_model_len": 32768, **extra}


# ------------------------------------------------------------------ inputs --


def _lengths(case):
    lo, hi, n = case["min_len"], case["max_len"], case["n_seq"]
    rng = random.Random(n * 1000003 + lo * 1009 + hi)
    return [rng.randint(lo, hi) for _ in range(n)]


def _blocks(tokens):
    return -(-tokens // PAGE)


def _tables(lengths, budget, inplace, g):
    """Source and destination pages.  Pages are scattered through the pool;
    the pages that compaction writes come together (the last ones, or in place
    the first ones), so that they can be returned as one view."""
    keep_pages = _blocks(budget) if budget else 0
    need = [_blocks(n) for n in lengths]
    n = len(lengths)
    if inplace:
        front = n * keep_pages
        rest = front + torch.randperm(sum(need) - front, generator=g)
        src, at = [], 0
        for i, c in enumerate(need):
            head = torch.arange(i * keep_pages, (i + 1) * keep_pages)
            src.append(torch.cat([head, rest[at : at + c - keep_pages]]))
            at += c - keep_pages
        return sum(need), src, None, (0, front)
    order = torch.randperm(sum(need), generator=g)
    src, at = [], 0
    for c in need:
        src.append(order[at : at + c])
        at += c
    out = sum(need) + torch.randperm(n * keep_pages, generator=g)
    dst = [out[i * keep_pages : (i + 1) * keep_pages] for i in range(n)] if budget else None
    return sum(need) + n * keep_pages, src, dst, (sum(need), sum(need) + n * keep_pages)


def _pool(case, n_caches, pages, seed, device):
    """[caches, pages, 128, kv, D] of normal values with a per-channel scale."""
    g = torch.Generator(device=device).manual_seed(seed)
    kv, d = case["kv"], case["head_dim"]
    pool = torch.empty((n_caches, pages, PAGE, kv, d), dtype=DTYPES[case["dtype"]], device=device)
    scale = 1.0 + 0.25 * torch.randn((n_caches, 1, 1, kv, d), generator=g, device=device)
    for i in range(n_caches):
        pool[i].normal_(generator=g)
        pool[i].mul_(scale[i].to(pool.dtype))
    return pool


def _omega(case, device):
    r = case["rotary"]
    return (1.0 / (case["theta"] ** (torch.arange(0, r, 2, dtype=torch.float32) / r))).to(device)


def _centres(case, g):
    """Query centres of one layer, per query head, on the host."""
    heads, freq, p = case["heads"], case["rotary"] // 2, case["head_dim"] - case["rotary"]
    qr = torch.randn(heads, freq, generator=g)
    qi = torch.randn(heads, freq, generator=g)
    qa = torch.sqrt(qr.square() + qi.square()) + torch.randn(heads, freq, generator=g).abs()
    qp = torch.randn(heads, p, generator=g) if p else None
    return qr, qi, qa, qp


def _layer_stats(case, seed, n, device):
    g = torch.Generator().manual_seed(seed)
    kv, qpk = case["kv"], case["heads"] // case["kv"]
    group = lambda t: None if t is None else t.view(kv, qpk, -1).contiguous().to(device)  # noqa: E731
    out = []
    for _ in range(n):
        qr, qi, qa, qp = _centres(case, g)
        out.append(DeviceLayerCalibrationStats(
            q_mean_real=group(qr), q_mean_imag=group(qi), q_abs_mean=group(qa),
            freq_scale_sq=torch.ones(kv, qpk, case["rotary"] // 2, device=device), omega=_omega(case, device),
            rope_style=case["style"], rotary_dim=case["rotary"], q_pass_mean=group(qp)))
    return out


def _select_options(case):
    return dict(budget=case["budget"], protected_prefix=case.get("prefix", 0), protected_recent=case["recent"],
                segments=case.get("segments", 8), policy=case.get("policy", "global"))


def _pipeline(case, stats, k, v, scoring, lengths):
    tables = ScoringTables.from_layer_stats(stats, build_geometric_offsets(case.get("max_model_len", 32768), k[0].device))
    options = _select_options(case) if "budget" in case else dict(
        budget=1, protected_prefix=0, protected_recent=0, segments=1, policy="global")
    return CompressionPipeline(
        scoring_k_caches=scoring, k_caches=k, v_caches=v, tables=tables, layer_aggregation="mean", max_seqs=len(lengths),
        max_seq_len=max(lengths), max_tokens=sum(lengths), score_aggregation=case.get("aggregation", "mean"),
        compaction_order="layer_major", **options)


def _prepare_cache(case, seed, device):
    lengths = _lengths(case)
    kind = case["kind"]
    budget = case.get("budget", 0)
    pages, src, dst, written = _tables(lengths, budget, case.get("inplace", False), torch.Generator().manual_seed(seed + 1))
    n_caches = case["layers"] * (1 if kind in ("score", "layer") else 2)
    pool = _pool(case, n_caches, pages, seed, device)
    src = [t.to(device) for t in src]
    dst = None if dst is None else [t.to(device) for t in dst]
    return lengths, pool, src, dst, written


def _prepare_score(case, seed, device):
    lengths, pool, src, _, _ = _prepare_cache(case, seed, device)
    layers = list(pool)
    stats = _layer_stats(case, seed + 2, case["layers"], device)
    pipeline = _pipeline(case, stats, layers, layers, layers, lengths)
    return {"pipeline": pipeline, "batch": Batch.build(device, lengths, lengths, src)}


def _prepare_step(case, seed, device):
    lengths, pool, src, dst, written = _prepare_cache(case, seed, device)
    k, v = list(pool[0::2]), list(pool[1::2])
    scoring = k[:: case["stride"]]
    stats = _layer_stats(case, seed + 2, len(scoring), device)
    pipeline = _pipeline(case, stats, k, v, scoring, lengths)
    batch = Batch.build(device, lengths, lengths, src, dst, budget=case["budget"])
    return {"pipeline": pipeline, "batch": batch, "rows": pool[:, written[0] : written[1]], "tokens": sum(lengths)}


def _prepare_compress(case, seed, device):
    lengths, pool, src, dst, written = _prepare_cache(case, seed, device)
    g = torch.Generator().manual_seed(seed + 2)
    partial = case["rotary"] != case["head_dim"]
    metadata = {"rope_style": case["style"], "head_dim": case["head_dim"], "rotary_dim": case["rotary"],
                "num_attention_heads": case["heads"], "num_kv_heads": case["kv"], "rope_theta": case["theta"],
                "model_type": "qwen2", "num_layers": case["layers"]}
    layers = {}
    for i in range(case["layers"]):
        qr, qi, qa, qp = _centres(case, g)
        layers[i] = {"q_mean_real": qr, "q_mean_imag": qi, "q_abs_mean": qa, "freq_scale_sq": torch.ones(1, qr.shape[1])}
        if qp is not None:
            layers[i]["q_pass_mean"] = qp
    model = ModelShape(model_type="qwen2", num_layers=case["layers"], num_attention_heads=case["heads"],
                       num_kv_heads=case["kv"], head_dim=case["head_dim"], rope_theta=case["theta"],
                       has_rope_scaling=False, rotary_dim=case["rotary"] if partial else None)
    options = {"kv_budget": case["budget"], "score_layer_stride": case["stride"],
               "protected_recent_window": case["recent"], "protected_prefix_window": case["prefix"],
               "position_policy": case["policy"], "position_segments": case["segments"],
               "score_aggregation": case["aggregation"]}
    config = SimpleNamespace(parallel_config=SimpleNamespace(tensor_parallel_size=1),
                             model_config=SimpleNamespace(max_model_len=case["max_model_len"]), speculative_config=None)
    # The layer order is a deployment's setting; "auto" would time trials inside the first calls.
    os.environ[COMPACTION_ORDER_ENV] = "layer_major"
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "stats.pt")
        torch.save({"metadata": metadata, "layer_stats": layers}, path)
        method = create_method("triattention", {"stats_path": path, **options}, config, model)
        caches = tuple(LayerCache("model.layers.%d.self_attn.attn" % i, i, pool[2 * i], pool[2 * i + 1])
                       for i in range(case["layers"]))
        method.bind_model_runner(SimpleNamespace(device=device), caches)
    requests = tuple(
        CompressionRequest(
            request_id="request-%d" % i, semantic_num_tokens=n, physical_num_tokens=n,
            source_block_ids=(tuple(src[i].tolist()),), destination_block_ids=(tuple(dst[i].tolist()),),
            source_block_ids_device=src[i], destination_block_ids_device=dst[i])
        for i, n in enumerate(lengths))
    return {"method": method, "requests": requests, "rows": pool[:, written[0] : written[1]], "tokens": sum(lengths)}


def _prepare_layer(case, seed, device):
    lengths, pool, src, _, _ = _prepare_cache(case, seed, device)
    (stats,) = _layer_stats(case, seed + 2, 1, device)
    n = lengths[0]
    qr, qi = stats.q_mean_real, stats.q_mean_imag
    offsets = build_geometric_offsets(case["max_model_len"], device)
    cos, sin = kernels.mean_phase_table(torch.tensor([n], device=device), offsets, stats.omega.view(1, -1))
    scale = torch.sqrt(stats.freq_scale_sq)
    extra = stats.q_abs_mean - torch.sqrt(qr.square() + qi.square() + 1e-8)
    out = torch.empty((case["kv"], case["heads"] // case["kv"], n), dtype=torch.float32, device=device)
    return {"args": (pool[0], src[0], qr, qi, scale, extra, cos.view(-1), sin.view(-1), n, out, PAGE, case["style"]),
            "kwargs": dict(q_pass_mean=stats.q_pass_mean, rotary_dim=case["rotary"]), "out": out}


def _scores(case, seed, device):
    """Aggregated scores as the scoring stage gives them: the mean over layers
    of the largest of a layer's standardised head scores."""
    g = torch.Generator(device=device).manual_seed(seed)
    total = sum(_lengths(case))
    return torch.randn(3, 8, total, generator=g, device=device).amax(1).mean(0)


def _prepare_select(case, seed, device):
    lengths = _lengths(case)
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    return {
        "args": (_scores(case, seed, device), torch.tensor(lengths, dtype=torch.int32, device=device),
                 torch.tensor(offsets, device=device), lengths,
                 torch.empty((len(lengths), case["budget"]), dtype=torch.int64, device=device)),
        "kwargs": dict(workspace=selection.select_workspace(len(lengths), case["segments"], case["policy"], device),
                       **_select_options(case)),
    }


def _prepare_compact(case, seed, device):
    lengths, pool, src, dst, written = _prepare_cache(case, seed, device)
    k, v = list(pool[0::2]), list(pool[1::2])
    stats = _layer_stats({**case, "style": "half"}, seed + 2, 1, device)
    pipeline = _pipeline(case, stats, k, v, k[:1], lengths)
    batch = Batch.build(device, lengths, lengths, src, dst, budget=case["budget"])
    # A keep set as selection leaves it: sorted, the recent window whole, the rest anywhere before it.
    g = torch.Generator(device=device).manual_seed(seed + 3)
    recent, budget = case["recent"], case["budget"]
    for i, n in enumerate(lengths):
        middle = torch.randperm(n - recent, generator=g, device=device)[: budget - recent].sort().values
        pipeline.keep[i] = torch.cat([middle, torch.arange(n - recent, n, device=device)])
    return {"pipeline": pipeline, "batch": batch, "rows": pool[:, written[0] : written[1]]}


def _prepare_calibrate(case, seed, device):
    g = torch.Generator(device=device).manual_seed(seed)
    shape = (case["layers"], case["tokens"], case["heads"] * case["head_dim"])
    rows = torch.empty(shape, dtype=DTYPES[case["dtype"]], device=device).normal_(mean=0.5, generator=g)
    return {"projected": list(rows), "shape": (case["heads"], case["head_dim"], case["rotary"])}


_PREPARE = {"step": _prepare_step, "compress": _prepare_compress, "score": _prepare_score, "layer": _prepare_layer,
            "select": _prepare_select, "compact": _prepare_compact, "calibrate": _prepare_calibrate}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, int(seed) * 16 + 1, torch.device("cuda", torch.cuda.current_device()))
    state["kind"] = case["kind"]
    return state


# -------------------------------------------------------------------- runs --


def _run_step(s):
    p = s["pipeline"]
    keep, tables, freed = p.step(s["batch"])
    return {"aggregate": p.agg[: s["tokens"]], "keep": keep, "tables": tables, "freed": freed, "rows": s["rows"]}


def _run_compress(s):
    results = s["method"].compress_batch(s["requests"])
    p = s["method"].pipeline
    return {"aggregate": p.agg[: s["tokens"]], "keep": p.keep[: len(results)], "rows": s["rows"],
            "kept": [r.physical_num_tokens for r in results]}


def _run_score(s):
    p, batch = s["pipeline"], s["batch"]
    p.score(batch)
    p.aggregate(batch)
    mean, var = p.head_statistics(batch)
    total = batch.total_tokens
    return {"aggregate": p.agg[:total], "raw": p.raw_scores()[:, :total], "mean": mean, "var": var}


def _run_layer(s):
    kernels.score_paged_keys_mean_precomputed(*s["args"], **s["kwargs"])
    return s["out"]


def _run_select(s):
    return selection.select_keep_indices_batched(*s["args"], **s["kwargs"])


def _run_compact(s):
    s["pipeline"].compact(s["batch"])
    return s["rows"]


def _run_calibrate(s):
    out = []
    for projected in s["projected"]:
        layer = calibration.LayerAccumulator()
        layer.add(projected, *s["shape"])
        out.append([layer.real_sum, layer.imag_sum, layer.abs_sum, layer.pass_sum])
    return out


_RUN = {"step": _run_step, "compress": _run_compress, "score": _run_score, "layer": _run_layer, "select": _run_select,
        "compact": _run_compact, "calibrate": _run_calibrate}


def run(state):
    return _RUN[state["kind"]](state)


# -------------------------------------------------------------------- work --


def work(case):
    kind = case["kind"]
    if kind == "calibrate":
        n = case["layers"] * case["tokens"] * case["heads"] * case["head_dim"]
        size = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": n * size, "flops": 4 * n}
    lengths = _lengths(case)
    total = sum(lengths)
    if kind == "select":
        return {"bytes": total * 4 + len(lengths) * case["budget"] * 8, "flops": 0}
    row = case["kv"] * case["head_dim"] * 2
    kept = case.get("budget", 0) * len(lengths)
    move = case["layers"] * kept * row * 4  # K and V, read and written
    if kind == "compact":
        return {"bytes": move + kept * 8, "flops": 0}
    # A token's score in one layer: every query head's product with the key
    # (per offset for "max") and with the magnitudes.
    layers = len(range(0, case["layers"], case.get("stride", 1)))
    n_off = case["max_model_len"].bit_length() if case["aggregation"] == "max" else 1
    rotary, rest = case["rotary"], case["head_dim"] - case["rotary"]
    flops = layers * total * case["heads"] * 2 * (rotary * n_off + rotary // 2 + rest)
    if kind == "layer":
        return {"bytes": total * row + total * case["heads"] * 4, "flops": flops}
    score = layers * total * row + total * 4
    if kind == "score":
        return {"bytes": score, "flops": flops}
    return {"bytes": score + total * 4 + kept * 8 + move, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("select", "compact"):
        return "exact"
    if kind == "calibrate":
        # Float32 terms (a rounded magnitude each), 64-bit sums.
        return {"rel": 1e-7, "max": 1e-5}
    if kind == "layer":
        return {"rel": 2e-5, "max": 2e-4}
    # Float32 scores and statistics; kept rows and indices can differ where two
    # scores at the threshold nearly tie.
    return {"rel": 2e-5, "max": 5e-4, "differ": 0.01}


# ------------------------------------------------------------------- exact --


def _exact_scores(case, key, stats, n, aggregation, offsets):
    """[heads, tokens] in float64 of keys [tokens, kv, D]; the phase argument
    is the float32 one that the scores are defined with."""
    f = case["rotary"] // 2
    key = key.double()
    rot = key[..., : 2 * f]
    kr, ki = (rot[..., 0::2], rot[..., 1::2]) if case["style"] == "interleaved" else (rot[..., :f], rot[..., f:])
    kr, ki = kr.permute(1, 0, 2).contiguous(), ki.permute(1, 0, 2).contiguous()  # [kv, tokens, F]
    qr, qi = stats.q_mean_real.double(), stats.q_mean_imag.double()
    a = torch.sqrt(stats.freq_scale_sq.double())
    # The magnitude coefficient is a float32 input of the scores.
    extra = (stats.q_abs_mean - torch.sqrt(stats.q_mean_real.square() + stats.q_mean_imag.square() + 1e-8)).double()
    angle = ((offsets + float(n)).unsqueeze(1) * stats.omega).double()
    cos, sin = torch.cos(angle), torch.sin(angle)
    if aggregation == "mean":
        cos, sin = cos.mean(0, keepdim=True), sin.mean(0, keepdim=True)
    best = None
    for c, s in zip(cos, sin):
        w_re, w_im = a * (qr * c - qi * s), a * (qi * c + qr * s)
        v = torch.bmm(w_re, kr.transpose(1, 2).contiguous()) + torch.bmm(w_im, ki.transpose(1, 2).contiguous())
        best = v if best is None else torch.maximum(best, v)
    mag = torch.sqrt(kr.square() + ki.square())
    out = best + torch.bmm(a * extra, mag.transpose(1, 2).contiguous())
    if stats.q_pass_mean is not None:
        rest = key[..., 2 * f :].permute(1, 2, 0).contiguous()
        out = out + torch.bmm(stats.q_pass_mean.double(), rest)
    return out.reshape(case["heads"], -1)


def _exact_aggregate(case, scoring, stats, src, lengths, device):
    offsets = build_geometric_offsets(case["max_model_len"], device)
    aggregate, raw, means, variances = [], [], [], []
    for i, n in enumerate(lengths):
        total, every, mean, var = 0.0, [], [], []
        for cache, layer in zip(scoring, stats):
            keys = cache[src[i]].reshape(-1, case["kv"], case["head_dim"])[:n]
            scores = _exact_scores(case, keys, layer, n, case["aggregation"], offsets)
            m, v = scores.mean(1), scores.var(1, correction=0)
            total = total + ((scores - m[:, None]) / v.clamp_min(1e-6).sqrt()[:, None]).amax(0)
            every.append(scores.t())
            mean.append(m)
            var.append(v)
        aggregate.append(total / len(stats))
        raw.append(torch.stack(every))
        means.append(torch.stack(mean))
        variances.append(torch.stack(var))
    return {"aggregate": torch.cat(aggregate), "raw": torch.cat(raw, 1), "mean": torch.stack(means, 1),
            "var": torch.stack(variances, 1)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("select", "compact"):
        return None
    seed, device = int(seed) * 16 + 1, torch.device("cuda", torch.cuda.current_device())
    if kind == "calibrate":
        state = _prepare_calibrate(case, seed, device)
        heads, dim, rotary = state["shape"]
        f, out = rotary // 2, []
        for rows in state["projected"]:
            q = rows.double().view(-1, heads, dim)
            re, im = q[..., :f], q[..., f:rotary]
            out.append([re.sum(0), im.sum(0), torch.sqrt(re.square() + im.square()).sum(0),
                        q[..., rotary:].sum(0) if rotary < dim else None])
        return out
    lengths, pool, src, _, _ = _prepare_cache(case, seed, device)
    if kind in ("score", "layer"):
        stats = _layer_stats(case, seed + 2, case["layers"], device)
        if kind == "layer":
            n = lengths[0]
            keys = pool[0][src[0]].reshape(-1, case["kv"], case["head_dim"])[:n]
            scores = _exact_scores(case, keys, stats[0], n, "mean", build_geometric_offsets(case["max_model_len"], device))
            return scores.view(case["kv"], -1, n)
        return _exact_aggregate(case, list(pool), stats, src, lengths, device)
    scoring = list(pool[0::2])[:: case["stride"]]
    if kind == "step":
        stats = _layer_stats(case, seed + 2, len(scoring), device)
    else:  # the calibration holds every layer
        stats = _layer_stats(case, seed + 2, case["layers"], device)[:: case["stride"]]
    return {"aggregate": _exact_aggregate(case, scoring, stats, src, lengths, device)["aggregate"]}
