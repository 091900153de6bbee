"""The workloads this package is timed on: one dict per case, inputs from a seed, one pass through the public API.

Paths (``case["path"]``) and what they stand for in a recommender's program:

* ``pooled``    EmbeddingBagCollection.forward on a KeyedJaggedTensor (serving lookups: fp32, bf16, int8 tables)
* ``features``  padded id matrices -> build_pooled_kjt (padding filtered) -> EmbeddingBagCollection.forward
* ``s_tokens``  FusedSequenceTokenizer.forward: behaviour-pool ids -> S-tokens of a OneTrans model
* ``ns_tokens`` FusedNSTokenizer.forward: scalar ids + dense features -> NS-tokens
* ``block``     OneTransBlock.forward, one interaction layer
* ``stack``     OneTransStack.forward, the whole backbone under the pyramid schedule
* ``train_pooled``  EmbeddingBagCollection forward + loss.backward() with the optimizer fused into the backward
* ``train_seq``     SequenceGather forward + loss.backward() with the optimizer fused into the backward
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch.distributed.optim import _apply_optimizer_in_backward

from __graft_entry__ import pdm_import

pdm = pdm_import()

ZIPF_SCATTER = 2654435761  # prime: rank -> row is a bijection, so hot rows are spread over the table
_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
_TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # online scoring of one request batch: the README's CPU-runnable collection, latency decides
        dict(name="pooled_fp32_b256", path="pooled", tables=8, rows_lo=100_000, rows_hi=100_000, dim=64, dtype="fp32",
             pooling="sum", out="fp32", batch=256, mean=10.0, lo=0, hi=50, alpha=0.0, index=64),
        # one id per categorical feature, tables from a thousand to forty million rows (a DLRM's sparse arch)
        dict(name="pooled_single_hot_bf16", path="pooled", tables=26, rows_lo=1_000, rows_hi=40_000_000, dim=128,
             dtype="bf16", pooling="sum", out="fp32", batch=65_536, mean=1.0, lo=1, hi=1, alpha=1.05, index=64),
        # quantized inference: int8 rows, multi-hot bags, the largest tables one GPU is asked to hold here
        dict(name="pooled_int8_mean", path="pooled", tables=64, rows_lo=5_000_000, rows_hi=5_000_000, dim=128,
             dtype="int8", pooling="mean", out="fp16", batch=16_384, mean=20.0, lo=1, hi=100, alpha=1.2, index=64),
        # a training or evaluation batch as the data loader leaves it: padded id matrices, 30 % padding
        dict(name="features_pooled_b8192", path="features", tables=26, rows=1_000_000, dim=64, dtype="bf16",
             pooling="mean", out="fp32", batch=8_192, length=20, pad=0.3, alpha=1.1),
        # S-tokens of the three behaviour pools (listen+, like, skip), item + artist + album per event
        dict(name="s_tokens_b1024", path="s_tokens", batch=1_024, pools=3, mean=150.0, max_len=256,
             item_rows=10_000_000, dims="256,64,64", d_model=256, dtype="bf16", alpha=1.1),
        # NS-tokens: uid / item / artist / album rows and four dense parts into 16 tokens of 256
        dict(name="ns_tokens_b1024", path="ns_tokens", batch=1_024, tables=4, rows=3_400_000, dim=64, dense=140,
             d_model=256, n_ns=16, dtype="bf16"),
        # the second layer of the 4-layer d 256 backbone on a full batch
        dict(name="block_d256_b1024", path="block", d_model=256, batch=1_024, s=384, n_ns=16, keep=256, ffn_mult=4),
        # the second layer of OneTransL on a full batch: 1500 S-tokens, 6 heads; the largest case
        dict(name="block_d384_b1024", path="block", d_model=384, batch=1_024, s=1_500, n_ns=16, keep=1_288, ffn_mult=4),
        # online scoring through the whole d 256 backbone
        dict(name="stack_d256_b16", path="stack", d_model=256, batch=16, s=384, n_ns=16, layers=4, keep_last=64,
             ffn_mult=4),
        # OneTransL scoring a small request batch through all eight layers
        dict(name="stack_d384_b8", path="stack", d_model=384, batch=8, s=1_500, n_ns=16, layers=8, keep_last=16,
             ffn_mult=4),
        # pooled lookups trained with Adam fused into the backward
        dict(name="train_pooled_adam", path="train_pooled", tables=8, rows=1_000_000, dim=64, pooling="sum",
             batch=16_384, mean=10.0, hi=50, optimizer="adam"),
        # sequence lookups trained with row-wise Adagrad fused into the backward (left padding reads row 0)
        dict(name="train_seq_adagrad", path="train_seq", batch=512, pools=3, mean=150.0, max_len=256,
             item_rows=1_000_000, dims="256,64,64", optimizer="rowwise_adagrad", alpha=1.1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["pooled", "features", "s_tokens", "ns_tokens", "block", "block", "stack", "stack",
                       "train_pooled", "train_seq"])
    if path == "pooled":
        tables, dim = rng.randint(1, 64), rng.choice([16, 32, 36, 64, 64, 100, 128, 128, 256])
        dtype = rng.choice(["fp32", "fp16", "bf16", "int8"])
        batch = _log(rng, 32, 65_536)
        single = rng.random() < 0.25
        mean = 1.0 if single else rng.uniform(2.0, 40.0)
        batch = max(32, min(batch, int(2e7 / (tables * mean))))
        lo = _log(rng, 1_000, 50_000)
        room = int(2e10 / (tables * (dim + 4 if dtype == "int8" else dim * _BYTES[dtype])))  # 20 GB of tables at most
        return dict(path=path, tables=tables, rows_lo=lo, rows_hi=min(room, _log(rng, 50_000, 5_000_000)), dim=dim,
                    dtype=dtype, pooling=rng.choice(["sum", "mean"]), out=rng.choice(["fp32", "fp16", "bf16"]),
                    batch=batch, mean=round(mean, 1), lo=1 if single else rng.choice([0, 1]),
                    hi=1 if single else 100, alpha=rng.choice([0.0, 1.05, 1.2]), index=rng.choice([32, 64]))
    if path == "features":
        tables, length = rng.randint(1, 26), rng.randint(1, 50)
        batch = max(32, min(_log(rng, 64, 65_536), int(2e7 / (tables * length))))
        return dict(path=path, tables=tables, rows=_log(rng, 1_000, 2_000_000), dim=rng.choice([16, 32, 64, 128]),
                    dtype=rng.choice(["fp32", "bf16"]), pooling=rng.choice(["sum", "mean"]), out="fp32", batch=batch,
                    length=length, pad=round(rng.uniform(0.0, 0.7), 2), alpha=rng.choice([0.0, 1.1]))
    if path in ("s_tokens", "train_seq"):
        max_len = rng.randint(16, 256)
        got = dict(path=path, batch=_log(rng, 8, 1_024 if path == "s_tokens" else 512), pools=rng.randint(1, 3),
                   mean=round(rng.uniform(0.2, 0.9) * max_len, 1), max_len=max_len,
                   item_rows=_log(rng, 20_000, 5_000_000 if path == "s_tokens" else 1_000_000),
                   dims=rng.choice(["256,64,64", "64,64,64", "128", "128,64", "64,64"]), alpha=rng.choice([0.0, 1.1]))
        if path == "s_tokens":
            got.update(d_model=rng.choice([128, 256, 384]), dtype=rng.choice(["bf16", "fp32"]))
        else:
            got.update(optimizer=rng.choice(["adam", "rowwise_adagrad"]))
        return got
    if path == "ns_tokens":
        return dict(path=path, batch=_log(rng, 8, 1_024), tables=rng.randint(0, 6), rows=_log(rng, 1_000, 3_000_000),
                    dim=rng.choice([32, 64]), dense=rng.randint(9, 260), d_model=rng.choice([128, 256, 384]),
                    n_ns=rng.choice([4, 8, 16]), dtype=rng.choice(["bf16", "fp32"]))
    if path == "train_pooled":
        tables = rng.randint(1, 12)
        batch = max(64, min(_log(rng, 64, 16_384), int(1.3e6 / (10 * tables))))
        return dict(path=path, tables=tables, rows=_log(rng, 2_000, 600_000), dim=rng.choice([16, 32, 64, 128]),
                    pooling=rng.choice(["sum", "mean"]), batch=batch, mean=round(rng.uniform(1.0, 12.0), 1), hi=50,
                    optimizer=rng.choice(["adam", "rowwise_adagrad"]))
    d_model, n_ns = rng.choice([128, 256, 256, 384, 384, 512]), rng.choice([5, 8, 16])
    s = _log(rng, 48, 1_500)
    got = dict(path=path, d_model=d_model, batch=1, s=s, n_ns=n_ns, ffn_mult=rng.choice([2, 4, 4]))
    if path == "block":
        got["keep"] = rng.randint(min(s, n_ns), s)
    else:
        got.update(layers=rng.randint(2, 8), keep_last=rng.randint(min(s, n_ns), s))
    one = work(got)["flops"]
    got["batch"] = max(1, min(_log(rng, 1, 1_024), int(4e12 / one)))
    return got


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------

def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _ids(g, n, rows, alpha):
    """``n`` row ids: uniform (``alpha`` 0) or Zipf(alpha) by inverting the continuous power law."""
    if alpha == 0.0:
        return torch.randint(0, rows, (n,), device="cuda", generator=g)
    u = torch.rand(n, device="cuda", dtype=torch.float64, generator=g)
    e = 1.0 - alpha
    r = ((rows ** e - 1.0) * u + 1.0).pow_(1.0 / e).floor_().clamp_(1, rows).to(torch.int64)
    return (r * ZIPF_SCATTER) % rows


def _lengths(g, n, mean, lo, hi):
    if lo == hi:
        return torch.full((n,), lo, dtype=torch.int64, device="cuda")
    return torch.poisson(torch.full((n,), mean, device="cuda"), generator=g).clamp_(lo, hi).to(torch.int64)


def _offsets(lengths):
    return torch.nn.functional.pad(lengths.cumsum(0), (1, 0))


def _table_rows(case):
    """Row counts of a pooled case's tables, log-uniform between its bounds (part of the model, not of the inputs)."""
    g = np.random.Generator(np.random.PCG64(7))
    lo, hi = math.log(case["rows_lo"]), math.log(case["rows_hi"])
    return [int(round(math.exp(lo + (hi - lo) * float(u)))) for u in g.random(case["tables"])]


def _ebc(case, rows, g, std=0.05):
    dt = {"fp32": pdm.DataType.FP32, "fp16": pdm.DataType.FP16, "bf16": pdm.DataType.BF16,
          "int8": pdm.DataType.INT8}[case.get("dtype", "fp32")]
    pool = pdm.PoolingType.SUM if case["pooling"] == "sum" else pdm.PoolingType.MEAN
    cfgs = [pdm.EmbeddingBagConfig(r, case["dim"], f"t{i}", dt, [f"f{i}"], pool,
                                   init_fn=lambda w: w.normal_(0.0, std, generator=g)) for i, r in enumerate(rows)]
    return pdm.EmbeddingBagCollection(cfgs, device=torch.device("cuda"), output_dtype=_TORCH[case.get("out", "fp32")])


def _seq_dims(case):
    return [int(d) for d in case["dims"].split(",")]


def _seq_inputs(case, g):
    """A batch of behaviour pools: flat ids per feature and lengths per pool, artist and album fixed by the item."""
    rows = _seq_rows(case)
    batch, groups = {}, {}
    for p in range(case["pools"]):
        mean = max(1.0, case["mean"] * (1.0, 0.3, 0.55)[p])
        lengths = _lengths(g, case["batch"], mean, 0, case["max_len"])
        n = int(lengths.sum())
        items = _ids(g, n, rows[0], case["alpha"])
        names = []
        for k, r in enumerate(rows):
            name = f"pool{p}_f{k}"
            batch[name] = items if k == 0 else (items * (40503, 69069)[k - 1] + 7) % r
            batch[name + "__lengths"] = lengths
            names.append(name)
        groups[f"pool{p}"] = names
    return batch, groups


def _seq_rows(case):
    return [case["item_rows"], max(1, case["item_rows"] // 10), max(1, case["item_rows"] // 5)][:len(_seq_dims(case))]


def _seq_collection(case, groups, g, dtype):
    cfgs = [pdm.EmbeddingConfig(r, d, f"t{k}", dtype, [fs[k] for fs in groups.values()],
                                init_fn=lambda w: w.normal_(0.0, 0.5, generator=g))
            for k, (r, d) in enumerate(zip(_seq_rows(case), _seq_dims(case)))]
    return pdm.EmbeddingCollection(cfgs, device=torch.device("cuda"))


def _fill(module, g, std=None):
    """Weights as trained bf16 checkpoints hold them: Xavier-sized normals (or ``std``), RMSNorm weights near one."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 1 and "norm" in name:
                p.normal_(1.0, 0.1, generator=g)
            else:
                s = std if std is not None else math.sqrt(2.0 / (p.shape[-1] + p.shape[-2]))
                p.normal_(0.0, s, generator=g)
            if "pos_emb" not in name and "norm" not in name:
                p.copy_(p.to(torch.bfloat16))
    return module.eval()


def _schedule(case):
    """S-tokens kept per layer, linear from all of them to ``keep_last``."""
    return pdm.pyramid_schedule(case["s"], case["keep_last"], case["layers"])


def _tag(collection, case):
    kw = {"lr": 0.01, "eps": 1e-8, "weight_decay": 1e-5}
    cls = torch.optim.Adam if case["optimizer"] == "adam" else pdm.RowWiseAdagrad
    for p in collection.parameters():
        _apply_optimizer_in_backward(cls, [p], kw)
    return collection


def prepare(case, seed):
    path, g = case["path"], _gen(seed)
    with torch.device("cuda"):
        if path == "pooled":
            rows, B = _table_rows(case), case["batch"]
            ebc = _ebc(case, rows, g)
            lengths = _lengths(g, len(rows) * B, case["mean"], case["lo"], case["hi"])
            per = lengths.view(len(rows), B).sum(1).tolist()
            values = torch.cat([_ids(g, n, r, case["alpha"]) for n, r in zip(per, rows)])
            values = values.to(torch.int32) if case["index"] == 32 else values
            return dict(case=case, ebc=ebc, values=values, offsets=_offsets(lengths),
                        keys=[f"f{i}" for i in range(len(rows))])
        if path == "features":
            rows = [case["rows"]] * case["tables"]
            ebc = _ebc(case, rows, g)
            feats = {}
            for i, r in enumerate(rows):
                ids = _ids(g, case["batch"] * case["length"], r - 1, case["alpha"]) + 1  # id 0 is the padding
                pad = torch.rand(ids.numel(), generator=g) < case["pad"]
                feats[f"f{i}"] = ids.masked_fill_(pad, 0).view(case["batch"], case["length"])
            return dict(case=case, ebc=ebc, feats=feats, keys=list(feats))
        if path == "s_tokens":
            batch, groups = _seq_inputs(case, g)
            ec = _seq_collection(case, groups, g, pdm.DataType.BF16 if case["dtype"] == "bf16" else pdm.DataType.FP32)
            K, d = sum(_seq_dims(case)), case["d_model"]
            toks = {n: _fill(pdm.SequentialTokenizer(K, d, max_len=2048), g, 0.05) for n in groups}
            return dict(case=case, batch=batch, tables=[ec.table_of(f) for f in next(iter(groups.values()))],
                        groups=groups, tok=pdm.FusedSequenceTokenizer(pdm.SequenceGather(ec, groups, case["max_len"]), toks))
        if path == "ns_tokens":
            names = [f"u{i}" for i in range(case["tables"])]
            dt = pdm.DataType.BF16 if case["dtype"] == "bf16" else pdm.DataType.FP32
            # one collection of scalar tables (uid, item, ...); a model without scalar ids keeps an unused one
            cfgs = [pdm.EmbeddingConfig(case["rows"], case["dim"], n, dt, [n],
                                        init_fn=lambda w: w.normal_(0.0, 0.5, generator=g)) for n in names or ["unused"]]
            ec = pdm.EmbeddingCollection(cfgs, device=torch.device("cuda"))
            widths = _dense_widths(case)
            K = case["tables"] * case["dim"] + sum(widths)
            tok = _fill(pdm.AutoSplitTokenizer(K, case["d_model"], case["n_ns"]), g, 0.05)
            batch = {n: torch.randint(0, case["rows"], (case["batch"],), generator=g) for n in names}
            dense = [torch.randn(case["batch"], w, generator=g) for w in widths]
            return dict(case=case, tok=pdm.FusedNSTokenizer(ec, names, tok), batch=batch, dense=dense,
                        tables=[ec.table_of(n) for n in names])
        if path in ("block", "stack"):
            D, n_ns = case["d_model"], case["n_ns"]
            if path == "block":
                model = pdm.OneTransBlock(D, D // 64, n_ns, case["ffn_mult"])
            else:
                model = pdm.OneTransStack(D, D // 64, n_ns, case["layers"], case["ffn_mult"], schedule=_schedule(case))
            x = torch.randn(case["batch"], case["s"] + n_ns, D, generator=g)
            return dict(case=case, model=_fill(model, g), x=x)
        if path == "train_pooled":
            rows, B = [case["rows"]] * case["tables"], case["batch"]
            ebc = _tag(_ebc(case, rows, g), case)
            lengths = _lengths(g, len(rows) * B, case["mean"], 0, case["hi"])
            values = _ids(g, int(lengths.sum()), case["rows"], 0.0)
            return dict(case=case, ebc=ebc, values=values, offsets=_offsets(lengths), keys=[f"f{i}" for i in range(len(rows))],
                        grad=torch.randn(B, case["tables"] * case["dim"], generator=g))
        batch, groups = _seq_inputs(case, g)
        ec = _tag(_seq_collection(case, groups, g, pdm.DataType.FP32), case)
        S, K = case["pools"] * case["max_len"], sum(_seq_dims(case))
        return dict(case=case, ec=ec, gather=pdm.SequenceGather(ec, groups, case["max_len"]), batch=batch, groups=groups,
                    grad=torch.randn(case["batch"], S, K, generator=g))


def _dense_widths(case):
    """The dense part in up to four pieces, as a model's dense features come (64, 6, 6 and the rest of 140)."""
    left, out = case["dense"], []
    for w in (64, 6, 6):
        if left > w + 1:
            out.append(w)
            left -= w
    return out + [left]


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------

def run(state):
    path = state["case"]["path"]
    if path == "train_pooled":
        ebc = state["ebc"]
        kjt = pdm.KeyedJaggedTensor(state["keys"], state["values"], offsets=state["offsets"])
        pooled = ebc(kjt).values()
        pooled.backward(state["grad"])
        fo = ebc.fused_optimizer
        return dict(pooled=pooled.detach(), weights=[ebc.embedding_bags[t.name].weight.detach()
                                                     for t in ebc.embedding_bag_configs()],
                    m1=fo.momentum1, m2=fo.momentum2)
    if path == "train_seq":
        ec = state["ec"]
        tokens, mask = state["gather"](state["batch"])
        tokens.backward(state["grad"])
        fo = ec.fused_optimizer
        return dict(tokens=tokens.detach(), mask=mask, weights=[ec.embeddings[t.name].weight.detach()
                                                                for t in ec.embedding_configs()],
                    m1=fo.momentum1, m2=fo.momentum2)
    with torch.no_grad():
        if path == "pooled":
            return state["ebc"](pdm.KeyedJaggedTensor(state["keys"], state["values"], offsets=state["offsets"])).values()
        if path == "features":
            kjt = pdm.kjt.build_pooled_kjt(state["feats"], state["keys"], 0)
            return dict(pooled=state["ebc"](kjt).values(), lengths=kjt.lengths(), offsets=kjt.offsets())
        if path == "s_tokens":
            tokens, mask = state["tok"](state["batch"])
            return dict(tokens=tokens, mask=mask)
        if path == "ns_tokens":
            return state["tok"](state["batch"], state["dense"])
        if path == "block":
            c = state["case"]
            return state["model"](state["x"], None, c["keep"] + c["n_ns"], c["s"])
        return state["model"](state["x"])


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------

def _distinct(n, rows, alpha):
    """Expected distinct rows among ``n`` ids of a table."""
    if n <= 0:
        return 0.0
    if alpha == 0.0:
        return rows * -math.expm1(-n / rows)
    e = 1.0 - alpha
    edges = np.unique(np.floor(np.geomspace(1, rows + 1, 4096)))
    mass = np.diff(edges ** e) / (rows ** e - 1.0)
    width = np.diff(edges)
    return float(min(n, np.sum(width * -np.expm1(-n * mass / width))))


def _layer_work(D, F, B, kv, q, n_ns):
    """(bytes, flops) of one block with its input and output in memory: K and V of every token, Q, out-projection and FFN
    of the kept ones, attention over the keys each query sees."""
    visible = q * (kv - q) + q * (q + 1) // 2
    flops = B * (4.0 * kv * D * D + 2.0 * q * D * D + 4.0 * D * visible + 2.0 * q * D * D + 4.0 * q * D * F)
    weights = 2.0 * (n_ns + 1) * (3 * D * D + 2 * D * F) + 2.0 * D * D
    return 4.0 * B * D * (kv + q) + weights, flops


def work(case):
    path, B = case["path"], case["batch"]
    if path == "pooled":
        rb = case["dim"] * _BYTES[case["dtype"]] if case["dtype"] != "int8" else case["dim"] + 4
        n = B * case["mean"]
        rows = sum(_distinct(n, r, case["alpha"]) for r in _table_rows(case))
        T = case["tables"]
        return dict(bytes=rows * rb + T * (n * case["index"] / 8 + B * 8 + B * case["dim"] * _BYTES[case["out"]]),
                    flops=T * n * case["dim"])
    if path == "features":
        T, n = case["tables"], B * case["length"]
        kept = n * (1.0 - case["pad"])
        rows = T * _distinct(kept, case["rows"], case["alpha"])
        rb = case["dim"] * _BYTES[case["dtype"]]
        return dict(bytes=rows * rb + T * (n * 8 + kept * 8 + B * 12 + B * case["dim"] * 4), flops=T * kept * case["dim"])
    if path in ("s_tokens", "train_seq"):
        dims, L, P = _seq_dims(case), case["max_len"], case["pools"]
        means = [min(L, max(1.0, case["mean"] * f)) for f in (1.0, 0.3, 0.55)[:P]]
        events = B * sum(means)
        rows = [min(_distinct(events, r, case["alpha"]), r) for r in _seq_rows(case)]
        K, slots = sum(dims), B * L * P
        ids = events * 8 * len(dims) + B * P * 8
        if path == "s_tokens":
            d = case["d_model"]
            return dict(bytes=ids + sum(r * w for r, w in zip(rows, dims)) * _BYTES[case["dtype"]] + slots * (4 * d + 1)
                        + P * (2 * (K * d + d * d + 2 * d) + 4 * L * d), flops=2.0 * events * (K * d + d * d))
        state = 16 if case["optimizer"] == "adam" else 0  # both moments read and written; row-wise: one word a row
        return dict(bytes=ids + slots * (4 * K + 1) + slots * 4 * K + sum(r * (w * (8 + state) + 8) for r, w in zip(rows, dims)),
                    flops=2.0 * slots * K)
    if path == "ns_tokens":
        K, N = case["tables"] * case["dim"] + case["dense"], case["d_model"] * case["n_ns"]
        return dict(bytes=B * (case["tables"] * (8 + case["dim"] * _BYTES[case["dtype"]]) + 4 * case["dense"])
                    + 2.0 * (K * N + N * N + 2 * N) + 4.0 * B * N, flops=2.0 * B * (K * N + N * N))
    if path == "train_pooled":
        n, T, dim = B * case["mean"], case["tables"], case["dim"]
        rows = T * _distinct(n, case["rows"], 0.0)
        state = 16 if case["optimizer"] == "adam" else 0
        return dict(bytes=T * (n * 8 + B * 8 + 2 * B * dim * 4) + rows * (dim * (8 + state) + 8), flops=2.0 * T * n * dim)
    D, F, kv, n_ns = case["d_model"], case["d_model"] * case["ffn_mult"], case["s"] + case["n_ns"], case["n_ns"]
    keeps = [case["keep"]] if path == "block" else _schedule(case)
    total_b = total_f = 0.0
    x_in = kv
    for keep in keeps:
        b, f = _layer_work(D, F, B, kv, keep + n_ns, n_ns)
        # the layers of a stack hand the residual stream on: only the first input and the last output are the path's
        total_b += b - 4.0 * B * D * (kv + keep + n_ns)
        total_f += f
        kv = keep + n_ns
    return dict(bytes=total_b + 4.0 * B * D * (x_in + kv), flops=total_f)


# ---------------------------------------------------------------------------------------------------------------
# exactness
# ---------------------------------------------------------------------------------------------------------------

def tolerance(case):
    """About four times the distance from 64 bits measured over the ranges above (in brackets)."""
    path = case["path"]
    if path in ("pooled", "features"):  # fp32 sums (1e-7); a 16-bit output is one rounding (fp16 2.1e-4, bf16 1.7e-3)
        return {"rel": {"fp32": 1e-6, "fp16": 8e-4, "bf16": 7e-3}[case["out"]]}
    if path in ("train_pooled", "train_seq"):  # fp32 sums and updates (2.2e-7); Adam divides by |g|, so an element whose
        return {"rel": 1e-6, "max": 0.02}      # gradient sums to nearly zero may move by any part of the step
    if path in ("s_tokens", "ns_tokens"):  # bf16 layers (3.6e-3)
        return {"rel": 0.014}
    return {"rel": 0.008 if path == "block" else 0.015}  # bf16 layers on an fp32 stream (block 1.9e-3, stack 3.7e-3)


def _pool64(tables, values, offsets, B, mean, dim):
    """Pooled rows in 64 bits; ``tables[t]`` maps ids to float64 rows."""
    outs = []
    bounds = offsets[::B].tolist()
    for t, rows_of in enumerate(tables):
        lens = offsets[t * B + 1:(t + 1) * B + 1] - offsets[t * B:(t + 1) * B]
        bag = torch.repeat_interleave(torch.arange(B, device="cuda"), lens)
        ids = values[bounds[t]:bounds[t + 1]].long()
        acc = torch.zeros(B, dim, dtype=torch.float64, device="cuda")
        for i in range(0, ids.numel(), 1 << 20):
            acc.index_add_(0, bag[i:i + (1 << 20)], rows_of(ids[i:i + (1 << 20)]))
        outs.append(acc / lens.clamp(min=1).unsqueeze(1) if mean else acc)
    return torch.cat(outs, 1)


def _rows64(weight, case):
    if case.get("dtype") != "int8":
        return lambda ids: weight.detach()[ids].double()

    def decode(ids):
        raw = weight[ids][:, :4 + case["dim"]].contiguous()
        sb = raw[:, :4].contiguous().view(torch.float16).double()
        return raw[:, 4:].double() * sb[:, :1] + sb[:, 1:]
    return decode


def _adam64(w, grad, touched):
    """First step of Adam with decoupled weight decay on the touched rows; betas as 32-bit numbers."""
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    m, v = (1 - b1) * grad, (1 - b2) * grad * grad
    step = 0.01 * ((m / (1 - b1)) / ((v / (1 - b2)).sqrt() + 1e-8) + 1e-5 * w)
    return torch.where(touched, w - step, w), torch.where(touched, m, 0.0 * m), torch.where(touched, v, 0.0 * v)


def _adagrad64(w, grad, touched):
    """First step of row-wise Adagrad with L2 weight decay."""
    g = grad + 1e-5 * w
    s = torch.where(touched.squeeze(1), (g * g).mean(1), 0.0)
    return torch.where(touched, w - 0.01 / (s.sqrt() + 1e-8).unsqueeze(1) * g, w), s


def _updated64(case, tables, grads, touched):
    """(weights, m1, m2) after the first fused step; Adam's moments laid out as the tables are, each 256-byte aligned."""
    weights, first, second = [], [], []
    for w, g, t in zip(tables, grads, touched):
        w = w.detach().double()
        if case["optimizer"] == "adam":
            w, m, v = _adam64(w, g, t.unsqueeze(1))
            if first and sum(x.numel() for x in first) % 64:
                gap = torch.zeros(-sum(x.numel() for x in first) % 64, dtype=torch.float64, device="cuda")
                first.append(gap)
                second.append(gap)
            first.append(m.flatten())
            second.append(v.flatten())
        else:
            w, s = _adagrad64(w, g, t.unsqueeze(1))
            first.append(s)
        weights.append(w)
    return weights, torch.cat(first), torch.cat(second) if second else None


def _rms64(x, w):
    return x * (x.pow(2).mean(-1, keepdim=True) + 1e-6).rsqrt() * w.double()


def _block64(blk, x, q_len, heads):
    """One OneTrans layer in 64 bits: shared weights on the S-tokens, per-token weights on the NS-tokens."""
    a, f = blk.attn, blk.ffn
    B, kv, D = x.shape
    n_ns = a.ns_qkv_weight.shape[0]

    def mixed(h, shared, own):
        n = h.shape[1] - n_ns
        return torch.cat([h[:, :n] @ shared.double().T, torch.matmul(h[:, n:].transpose(0, 1), own.double().transpose(1, 2)
                                                                     ).transpose(0, 1)], 1)

    qkv = mixed(_rms64(x, blk.norm1.weight), a.s_qkv.weight, a.ns_qkv_weight).view(B, kv, 3, heads, D // heads)
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    s = torch.matmul(q[:, :, kv - q_len:], k.transpose(-1, -2)) / math.sqrt(D // heads)
    see = torch.arange(kv, device="cuda") <= torch.arange(q_len, device="cuda").unsqueeze(1) + (kv - q_len)
    o = torch.matmul(torch.softmax(s.masked_fill(~see, float("-inf")), -1), v)
    z = o.transpose(1, 2).reshape(B, q_len, D) @ a.out_proj.weight.double().T + x[:, kv - q_len:]
    u = torch.nn.functional.gelu(mixed(_rms64(z, blk.norm2.weight), f.s_w1.weight, f.ns_w1))
    return z + mixed(u, f.s_w2.weight, f.ns_w2)


def _mlp64(x, proj):
    h = torch.nn.functional.gelu(x @ proj[0].weight.double().T + proj[0].bias.double())
    return h @ proj[2].weight.double().T + proj[2].bias.double()


def _padded_ids(case, state, feature):
    """[B, S] ids of the feature-th feature, each pool left padded with id 0, and the mask of real events."""
    ids, mask, B, L = [], [], case["batch"], case["max_len"]
    for names in state["groups"].values():
        flat, lengths = state["batch"][names[feature]], state["batch"][names[feature] + "__lengths"]
        start = _offsets(lengths)[:-1].unsqueeze(1)
        kept = lengths.clamp(max=L).unsqueeze(1)
        slot = torch.arange(L, device="cuda").unsqueeze(0) - (L - kept)
        real = slot >= 0
        at = (start + lengths.unsqueeze(1) - kept + slot).clamp(0, max(flat.numel() - 1, 0))
        ids.append(torch.where(real, flat[at] if flat.numel() else torch.zeros_like(at), 0))
        mask.append(real)
    return torch.cat(ids, 1), torch.cat(mask, 1)


@torch.no_grad()
def exact(case, seed):
    path = case["path"]
    with torch.enable_grad():  # tagging an embedding weight with its optimizer needs its autograd node
        s = prepare(case, seed)
    if path in ("pooled", "features"):
        B, T = case["batch"], case["tables"]
        tables = [_rows64(s["ebc"].embedding_bags[f"t{i}"].weight, case) for i in range(T)]
        if path == "pooled":
            return _pool64(tables, s["values"], s["offsets"], B, case["pooling"] == "mean", case["dim"])
        kept = torch.stack([m.ne(0) for m in s["feats"].values()])
        lengths = kept.sum(2).flatten()
        values = torch.cat([m[m.ne(0)] for m in s["feats"].values()])
        pooled = _pool64(tables, values, _offsets(lengths), B, case["pooling"] == "mean", case["dim"])
        return dict(pooled=pooled, lengths=None, offsets=None)
    if path == "s_tokens":
        ids = [_padded_ids(case, s, k) for k in range(len(s["tables"]))]
        raw_of = lambda lo, hi, cols: torch.cat([t.detach()[i[0][lo:hi, cols]] for t, i in zip(s["tables"], ids)], -1).double()  # noqa: E731
        L, out = case["max_len"], []
        for p, name in enumerate(s["groups"]):
            tok, parts = s["tok"].tokenizers[name], []
            for lo in range(0, case["batch"], 64):
                y = _mlp64(raw_of(lo, lo + 64, slice(p * L, (p + 1) * L)), tok.proj)
                parts.append(y + tok.pos_emb.weight[:L].double())
            out.append(torch.cat(parts))
        return dict(tokens=torch.cat(out, 1), mask=None)
    if path == "ns_tokens":
        rows = [t.detach()[s["batch"][f"u{i}"]].double() for i, t in enumerate(s["tables"])]
        x = torch.cat(rows + [d.double() for d in s["dense"]], 1)
        return _mlp64(x, s["tok"].tokenizer.proj).view(case["batch"], case["n_ns"], case["d_model"])
    if path in ("block", "stack"):
        heads, out = case["d_model"] // 64, []
        blocks = [s["model"]] if path == "block" else list(s["model"].blocks)
        keeps = [case["keep"]] if path == "block" else _schedule(case)
        chunk = max(1, int(2e9 / (8.0 * heads * (case["s"] + case["n_ns"]) ** 2)))
        for lo in range(0, case["batch"], chunk):
            x = s["x"][lo:lo + chunk].double()
            for blk, keep in zip(blocks, keeps):
                x = _block64(blk, x, keep + case["n_ns"], heads)
            out.append(x)
        return torch.cat(out)
    if path == "train_pooled":
        B, T, dim, mean = case["batch"], case["tables"], case["dim"], case["pooling"] == "mean"
        tables = [s["ebc"].embedding_bags[f"t{i}"].weight.detach() for i in range(T)]
        pooled = _pool64([_rows64(w, {}) for w in tables], s["values"], s["offsets"], B, mean, dim)
        bounds, grads, touched = s["offsets"][::B].tolist(), [], []
        for t, w in enumerate(tables):
            lens = s["offsets"][t * B + 1:(t + 1) * B + 1] - s["offsets"][t * B:(t + 1) * B]
            bag = torch.repeat_interleave(torch.arange(B, device="cuda"), lens)
            ids = s["values"][bounds[t]:bounds[t + 1]]
            gt = s["grad"][:, t * dim:(t + 1) * dim].double()
            gt = gt / lens.clamp(min=1).unsqueeze(1) if mean else gt
            grads.append(torch.zeros(w.shape, dtype=torch.float64, device="cuda").index_add_(0, ids, gt[bag]))
            touched.append(torch.zeros(w.shape[0], dtype=torch.bool, device="cuda").index_fill_(0, ids, True))
        weights, m1, m2 = _updated64(case, tables, grads, touched)
        return dict(pooled=pooled, weights=weights, m1=m1, m2=m2)
    names = next(iter(s["groups"].values()))
    tables = [s["ec"].table_of(f).detach() for f in names]
    grads, touched, tokens, col = [], [], [], 0
    for k, (w, d) in enumerate(zip(tables, _seq_dims(case))):
        ids, _ = _padded_ids(case, s, k)
        tokens.append(w[ids].double())
        gt = s["grad"][:, :, col:col + d].reshape(-1, d).double()
        real = ids.flatten().ne(0)  # most slots are padding and read row 0: its gradient is summed by itself
        grads.append(torch.zeros(w.shape, dtype=torch.float64, device="cuda").index_add_(0, ids.flatten()[real], gt[real]))
        grads[-1][0] = gt[~real].sum(0)
        touched.append(torch.zeros(w.shape[0], dtype=torch.bool, device="cuda").index_fill_(0, ids.flatten(), True))
        col += d
    weights, m1, m2 = _updated64(case, tables, grads, touched)
    return dict(tokens=torch.cat(tokens, -1), mask=None, weights=weights, m1=m1, m2=m2)
