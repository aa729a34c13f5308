"""Performance cases: the work a user of the library has it do, through its public entry points.

Two groups, as in the programs that use the library:

  * the training loop, one call (or one layer) per minibatch: fused decode + mean aggregation of affine, log-domain,
    VQ and two-table features, the unfused form of the same (row fetch, decode, aggregate), and the first GraphSAGE
    layer forward and backward over a compression manager;
  * the offline encoder, once per feature table: scalar codes with their statistics, codebook training, VQ codes, and
    nearest-centre assignment.

`listed()` names twelve of them, `draw()` gives others of the same ranges.  Every case is a dict of plain values;
`prepare` makes from it what the caller has in hand (tables, graph, codebooks, layers) on the GPU, and `run` makes one
pass.
"""
import math

import numpy as np
import torch

import f2cgt_amd
from f2cgt_amd import pipeline, synth

_DTYPES = {"int64": torch.int64, "int32": torch.int32}


# ---- the cases ------------------------------------------------------------------------------------
def listed():
    return [
        # one minibatch of the training loop: 1024 seed nodes with their own 4-bit table, their sampled neighbours in a
        # 32-columns-per-byte VQ table, layer forward and backward.  Launches and host time count here.
        {"name": "layer_minibatch", "kind": "layer", "nodes": 1000000, "seeds": 20000, "batch": 1024, "dst": 1024,
         "fanout": 10, "dim": 128, "width": 32, "seed_bits": 4, "hidden": 256},
        # the smallest aggregation: 8-bit codes, a block of 1e4 rows
        {"name": "affine8_small", "kind": "affine", "bits": 8, "nodes": 100000, "dim": 128, "rows": 10000,
         "degree": "fixed", "fanout": 10, "ids": "uniform", "zipf": 0.0, "index": "int64"},
        # an ordinary one: 4-bit codes, power-law degrees, skewed ids, 100 columns
        {"name": "affine4_powerlaw", "kind": "affine", "bits": 4, "nodes": 2400000, "dim": 100, "rows": 250000,
         "degree": "powerlaw", "fanout": 12, "ids": "zipf", "zipf": 1.1, "index": "int64"},
        # the encoder's default ratio, 1-bit log-domain codes, at Reddit's odd width and with ragged rows
        {"name": "sq1_reddit", "kind": "sq", "bits": 1, "nodes": 232965, "dim": 602, "rows": 60001,
         "degree": "ragged", "fanout": 20, "ids": "uniform", "zipf": 0.0, "index": "int32"},
        # vector codes of a 1e7-node graph, 15 neighbours per row
        {"name": "vq_16x8", "kind": "vq", "nodes": 10000000, "codebooks": 16, "width": 8, "dim": 128, "rows": 500000,
         "degree": "fixed", "fanout": 15, "ids": "zipf", "zipf": 1.1, "index": "int64"},
        # the widest features and the largest output: 768 columns, 24 codebooks
        {"name": "vq_24x32", "kind": "vq", "nodes": 240000000, "codebooks": 24, "width": 32, "dim": 768,
         "rows": 600000, "degree": "fixed", "fanout": 10, "ids": "zipf", "zipf": 1.1, "index": "int64"},
        # hot rows in an 8-bit table, the others in a VQ table, 1e8 nodes
        {"name": "hybrid", "kind": "hybrid", "nodes": 100000000, "hot": 0.05, "codebooks": 8, "width": 16, "dim": 128,
         "rows": 1000000, "degree": "fixed", "fanout": 12, "ids": "zipf", "zipf": 1.2, "index": "int64"},
        # the unfused form: source rows fetched from the table, decoded, averaged
        {"name": "unfused_vq", "kind": "unfused", "method": "vq", "bits": 0, "nodes": 2400000, "width": 16, "dim": 128,
         "sources": 200000, "rows": 30000, "degree": "ragged", "fanout": 15, "index": "int64"},
        # offline: scalar codes of a feature table, statistics and codes
        {"name": "encode_sq4", "kind": "encode_sq", "nodes": 120000, "dim": 100, "bits": 4, "sample": 120000},
        # offline: codebook training of a 96-column table, six slices of 16 columns, from a sample of 150 000 rows; the
        # trainer is held to eight steps (it takes about forty to its own end): further on the rows at near-ties decide
        # where the centres go, and two correct runs drift apart
        {"name": "train_vq", "kind": "train_vq", "nodes": 200000, "dim": 96, "width": 16, "centers": 256,
         "sample": 150000, "steps": 8},
        # offline: VQ codes of a feature table, 16 columns per code byte
        {"name": "encode_vq", "kind": "encode_vq", "nodes": 500000, "dim": 128, "width": 16, "centers": 256},
        # nearest-centre assignment of one wide slice (squared L2)
        {"name": "assign_32", "kind": "assign", "rows": 1000000, "dim": 32, "centers": 256, "metric": "l2"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng):
    """Feature widths of the usual graph data sets, and any other."""
    return rng.choice([100, 128, 256, 300, 500, 602, 2 * rng.randint(24, 150), rng.randint(48, 300)])


def _graph(rng, max_rows, max_edges):
    """Degree law and sizes of a block: R rows and about E edges at most."""
    rows = _log(rng, 1000, max_rows)
    degree = rng.choice(["fixed", "ragged", "powerlaw"])
    fanout = rng.randint(2, 25)
    mean = {"fixed": fanout, "ragged": fanout / 2, "powerlaw": 2.5}[degree]
    rows = max(500, min(rows, int(max_edges / mean)))
    ids = rng.choice(["uniform", "zipf"])
    return {"rows": rows, "degree": degree, "fanout": fanout, "ids": ids,
            "zipf": round(rng.uniform(1.05, 1.25), 2) if ids == "zipf" else 0.0, "index": rng.choice(["int64", "int64", "int32"])}


def draw(rng):
    kind = rng.choice(["layer", "affine", "affine", "sq", "sq", "vq", "vq", "hybrid", "unfused", "encode_sq", "train_vq",
                       "encode_vq", "assign"])
    case = {"kind": kind}
    if kind == "layer":
        batch = _log(rng, 500, 4000)
        case.update(nodes=_log(rng, 200000, 4000000), seeds=_log(rng, 10000, 100000), batch=batch,
                    dst=batch * rng.choice([1, 1, 4, 8]), fanout=rng.randint(5, 20), dim=rng.choice([96, 100, 128, 256]),
                    width=rng.choice([16, 32]), seed_bits=rng.choice([4, 8]), hidden=rng.choice([128, 256]))
    elif kind == "affine":
        dim = _width(rng)
        case.update(bits=rng.choice([4, 8]), nodes=_log(rng, 30000, 2400000 * 100 // dim), dim=dim)
        case.update(_graph(rng, 25000000 // dim, 250000000 // dim))
    elif kind == "sq":
        dim = _width(rng)
        case.update(bits=rng.choice([1, 1, 2, 4, 8]), nodes=_log(rng, 30000, 2400000 * 100 // dim), dim=dim)
        case.update(_graph(rng, 40000000 // dim, 400000000 // dim))
    elif kind == "vq":
        width = rng.choice([8, 16, 32])
        books = rng.randint(max(2, 64 // width), 768 // width)
        dim = books * width - rng.choice([0, 0, 0, rng.randint(1, width // 2)])
        case.update(nodes=_log(rng, 100000, 30000000), codebooks=books, width=width, dim=dim)
        case.update(_graph(rng, 200000000 // dim, 1500000000 // dim))
    elif kind == "hybrid":
        books, width = rng.choice([(8, 16), (16, 8), (8, 32), (13, 8), (6, 16)])
        case.update(nodes=_log(rng, 1000000, 50000000), hot=round(rng.uniform(0.02, 0.2), 3), codebooks=books, width=width,
                    dim=books * width)
        case.update(_graph(rng, 60000000 // (books * width), 600000000 // (books * width)))
        case.update(ids="zipf", zipf=round(rng.uniform(1.05, 1.25), 2))
    elif kind == "unfused":
        method = rng.choice(["sq", "vq"])
        rows = _log(rng, 1000, 60000)
        case.update(method=method, bits=rng.choice([1, 4, 8]) if method == "sq" else 0, nodes=_log(rng, 200000, 4000000),
                    width=rng.choice([8, 16, 32]), dim=rng.choice([100, 128, 256, 2 * rng.randint(24, 150)]),
                    sources=rows * rng.randint(2, 7), rows=rows, degree=rng.choice(["fixed", "ragged"]),
                    fanout=rng.randint(5, 20), index=rng.choice(["int64", "int32"]))
    elif kind == "encode_sq":
        dim = _width(rng)
        nodes = min(_log(rng, 20000, 150000), 12000000 // dim)
        case.update(nodes=nodes, dim=dim, bits=rng.choice([1, 2, 4, 8, 16]), sample=max(2000, int(nodes * rng.uniform(0.5, 1.0))))
    elif kind == "train_vq":
        width = rng.choice([8, 16, 32])
        nodes = _log(rng, 50000, 200000)
        case.update(nodes=nodes, dim=rng.randint(width, 96), width=width, centers=rng.choice([64, 128, 256]),
                    sample=max(20000, int(nodes * 0.75)), steps=8)
    elif kind == "encode_vq":
        width = rng.choice([8, 16, 32])
        dim = rng.randint(40, 256)
        case.update(nodes=_log(rng, 50000, 64000000 // dim), dim=dim, width=width, centers=rng.choice([64, 128, 256]))
    else:
        case.update(rows=_log(rng, 20000, 1000000), dim=rng.choice([8, 16, 32, rng.randint(4, 48)]),
                    centers=rng.choice([64, 128, 256, rng.randint(16, 256)]), metric=rng.choice(["l2", "cosine"]))
    return case


# ---- inputs ---------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _ids(case, n_ids, size, g, dtype):
    if case.get("ids") == "zipf":
        return synth.zipf_ids(n_ids, (size,), case["zipf"], g, "cuda", dtype)
    return torch.randint(0, n_ids, (size,), generator=g, device="cuda").to(dtype)


def _degrees(case, rows, g):
    if case["degree"] == "fixed":
        return torch.full((rows,), case["fanout"], dtype=torch.int64, device="cuda")
    if case["degree"] == "ragged":      # a sampler's block: up to `fanout` neighbours, none for an isolated node
        return torch.randint(0, case["fanout"] + 1, (rows,), generator=g, device="cuda")
    return synth.powerlaw_degrees(rows, 2.1, max(2, case["fanout"]), g, "cuda")


def _block(case, n_src, g):
    """indptr, indices of a sampled block over n_src source rows."""
    dtype = _DTYPES[case["index"]]
    deg = _degrees(case, case["rows"], g)
    indptr = synth.csc_from_degrees(deg, dtype)
    return indptr, _ids(case, n_src, int(deg.sum().item()), g, dtype)


def _affine_table(nodes, dim, bits, g):
    """Codes and column parameters of normal features with a scale of their own per column, quantised in chunks
    between the extremes that a sample of that size has."""
    scale_c = 0.5 + 1.5 * torch.rand((dim,), generator=g, device="cuda")
    sample = torch.randn((min(nodes, 200000), dim), generator=g, device="cuda") * scale_c
    _, params = synth.affine_quantise(sample, bits)
    del sample
    per = 8 // bits
    table = torch.empty((nodes, (dim + per - 1) // per), dtype=torch.uint8, device="cuda")
    step = max(1, 40000000 // dim)
    for lo in range(0, nodes, step):
        x = torch.randn((min(step, nodes - lo), dim), generator=g, device="cuda") * scale_c
        q = torch.round((x - params[0]) / params[1]).clamp_(0, (1 << bits) - 1).to(torch.uint8)
        table[lo:lo + q.shape[0]] = synth.pack_low_first(q, bits) if bits < 8 else q
    return table, params


def _features(nodes, dim, g):
    """Feature rows with some structure: a mixture of 64 directions plus noise, column scales apart."""
    hubs = torch.randn((64, dim), generator=g, device="cuda")
    pick = torch.randint(0, 64, (nodes,), generator=g, device="cuda")
    scale_c = 0.5 + 1.5 * torch.rand((dim,), generator=g, device="cuda")
    return (0.6 * hubs[pick] + torch.randn((nodes, dim), generator=g, device="cuda")) * scale_c


def _sq_codebook(dim, g):
    """One log-domain codebook (fmin, fmax, emin, emax, mean) over all columns, as normal features have it."""
    spread = float(0.8 + 0.4 * torch.rand((1,), generator=g, device="cuda").item())
    fmin, fmax = 0.006 * spread, 2.8 * spread
    return torch.tensor([[fmin, fmax, math.log2(fmin), math.log2(fmax) + 1e-5, 0.8 * spread]], device="cuda")


def _sq_table(nodes, dim, bits, g):
    """Log-domain codes in storage form: packed int8 for up to 8 bits."""
    return torch.randint(-128, 128, (nodes, (dim * bits + 7) // 8), generator=g, device="cuda", dtype=torch.int8)


def _vq_table(nodes, books, width, g):
    codes = torch.randint(0, 256, (nodes, books), generator=g, device="cuda", dtype=torch.uint8)
    return codes, torch.randn((books, 256, width), generator=g, device="cuda")


def _slice8(dim):
    """Columns per log-domain codebook of one codebook for all columns (a multiple of eight)."""
    return (dim + 7) // 8 * 8


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    capi = f2cgt_amd.load()
    s = {"kind": kind, "capi": capi, "case": case}
    if kind == "affine":
        s["table"], s["params"] = _affine_table(case["nodes"], case["dim"], case["bits"], g)
        s["indptr"], s["indices"] = _block(case, case["nodes"], g)
    elif kind == "sq":
        s["table"], s["books"] = _sq_table(case["nodes"], case["dim"], case["bits"], g), _sq_codebook(case["dim"], g)
        s["indptr"], s["indices"] = _block(case, case["nodes"], g)
    elif kind == "vq":
        s["table"], s["books"] = _vq_table(case["nodes"], case["codebooks"], case["width"], g)
        s["indptr"], s["indices"] = _block(case, case["nodes"], g)
    elif kind == "hybrid":
        wl = synth.c4_hybrid("cuda", _DTYPES[case["index"]], case["nodes"], case["dim"], case["hot"], case["codebooks"], 256,
                             case["width"], 1000, 1, case["zipf"], seed)
        s.update({k: wl[k] for k in ("row_map", "sq_codes", "sq_params", "vq_codes", "vq_codebooks")})
        s["indptr"], s["indices"] = _block(case, case["nodes"], g)
    elif kind == "unfused":
        books = (case["dim"] + case["width"] - 1) // case["width"]
        if case["method"] == "vq":
            table, cb = _vq_table(case["nodes"], books, case["width"], g)
            config = (case["width"], -1)
        else:
            table, cb = _sq_table(case["nodes"], case["dim"], case["bits"], g), _sq_codebook(case["dim"], g)
            config = (_slice8(case["dim"]), case["bits"])
        s["manager"] = pipeline.CompressionManager({"methods": [case["method"]], "feat_dim": case["dim"], "configs": [config],
                                                    "codebooks": [cb], "compression_data": table}, fusion=False)
        s["nodes"] = torch.randperm(case["nodes"], generator=g, device="cuda")[:case["sources"]].clone()
        s["indptr"], s["indices"] = _block(case, case["sources"], g)
    elif kind == "layer":
        dim, width = case["dim"], case["width"]
        table, cb = _vq_table(case["nodes"], (dim + width - 1) // width, width, g)
        seeds = torch.randperm(case["nodes"], generator=g, device="cuda")[:case["seeds"]].clone()
        s["manager"] = pipeline.CompressionManager(
            {"methods": ["sq", "vq"], "feat_dim": dim, "configs": [(_slice8(dim), case["seed_bits"]), (width, -1)],
             "codebooks": [_sq_codebook(dim, g), cb], "compression_data": table,
             "seeds_compression_data": _sq_table(case["seeds"], dim, case["seed_bits"], g), "seeds": seeds}, fusion=True)
        torch.manual_seed(seed)
        s["layer"] = pipeline.MySAGEConv(dim, case["hidden"], "mean", s["manager"], activation=torch.relu).cuda()
        # a sampler's block: batch nodes first, then the other destination nodes, then the nodes only read
        deg = torch.randint(1, case["fanout"] + 1, (case["dst"],), generator=g, device="cuda")
        s["indptr"] = synth.csc_from_degrees(deg, torch.int64)
        edges = int(deg.sum().item())
        n_src = case["dst"] + edges // 2
        s["batch"] = seeds[torch.randperm(case["seeds"], generator=g, device="cuda")[:case["batch"]]].clone()
        rest = torch.randint(0, case["nodes"], (n_src - case["batch"],), generator=g, device="cuda")
        s["nodes"] = torch.cat([s["batch"], rest])
        s["indices"] = torch.randint(0, n_src, (edges,), generator=g, device="cuda")
        s["grad"] = torch.randn((case["dst"], case["hidden"]), generator=g, device="cuda")
    elif kind == "encode_sq":
        s["features"] = _features(case["nodes"], case["dim"], g)
        s["sample"] = torch.randperm(case["nodes"], generator=g, device="cuda")[:case["sample"]].clone()
    elif kind == "train_vq":
        s["features"] = _features(case["nodes"], case["dim"], g)
        s["sample"] = torch.randperm(case["nodes"], generator=g, device="cuda")[:case["sample"]].clone()
        s["seed"] = seed
    elif kind == "encode_vq":
        s["features"] = _features(case["nodes"], case["dim"], g)
        books = (case["dim"] + case["width"] - 1) // case["width"]
        # centres as training leaves them: near the data, the unused columns of the last slice zero
        rows = torch.randperm(case["nodes"], generator=g, device="cuda")[:case["centers"]]
        cb = torch.zeros((books, case["centers"], case["width"]), device="cuda")
        for i in range(books):
            part = s["features"][rows, i * case["width"]:min((i + 1) * case["width"], case["dim"])]
            cb[i, :, :part.shape[1]] = pipeline.normalize(part)
        s["books"] = cb
    else:
        s["x"] = torch.randn((case["rows"], case["dim"]), generator=g, device="cuda")
        s["centers"] = torch.randn((case["centers"], case["dim"]), generator=g, device="cuda")
    return s


# ---- one pass -------------------------------------------------------------------------------------
def run(s):
    capi, case, kind = s["capi"], s["case"], s["kind"]
    if kind == "affine":
        return capi.sq_affine_decompress_spmm_csr(s["table"], s["params"], s["indptr"], s["indices"], case["bits"], case["dim"])
    if kind == "sq":
        return capi.sq_decompress_spmm_csr(s["table"], s["books"], s["indptr"], s["indices"], case["bits"],
                                           _slice8(case["dim"]), case["dim"])
    if kind == "vq":
        return capi.vq_decompress_spmm_csr(s["table"], s["books"], s["indptr"], s["indices"], case["dim"])
    if kind == "hybrid":
        return capi.hybrid_decompress_spmm_csr(s["row_map"], s["sq_codes"], s["sq_params"], s["vq_codes"], s["vq_codebooks"],
                                               s["indptr"], s["indices"], case["dim"])
    if kind == "unfused":
        decoded = s["manager"].get_all_data(s["nodes"])
        return decoded, capi.spmm_csr(decoded, s["indptr"], s["indices"])
    if kind == "layer":
        sm, layer = s["manager"], s["layer"]
        seeds_feature = sm.get_seeds_data(s["batch"])
        all_feature = sm.get_all_data(s["nodes"])
        h_self = sm.reorganize_seeds_data(seeds_feature, all_feature, case["dst"])
        layer.zero_grad(set_to_none=True)
        h = layer((s["indptr"], s["indices"]), (h_self, all_feature))
        h.backward(s["grad"])
        return h.detach(), [p.grad for p in layer.parameters()]
    if kind == "encode_sq":
        return pipeline.sq_compress(s["features"], case["bits"], _slice8(case["dim"]), sample_index=s["sample"])
    if kind == "train_vq":
        torch.manual_seed(s["seed"])     # the trainer draws its first centres: a repeatable run seeds them
        return pipeline.vq_metadata(s["features"], case["centers"], case["width"], sample_index=s["sample"],
                                    max_iter=case["steps"])
    if kind == "encode_vq":
        return pipeline.vq_compress(s["features"], case["centers"], case["width"], codebooks=s["books"])
    return capi.vq_encode(s["x"], s["centers"], case["metric"])


# ---- what a pass cannot do without ------------------------------------------------------------------
def _mean_degree(case):
    if case["degree"] == "fixed":
        return float(case["fanout"])
    if case["degree"] == "ragged":
        return case["fanout"] / 2.0
    cap = max(2, case["fanout"])
    d = np.arange(1, cap, dtype=np.float64)
    tail = np.arange(cap, 100000, dtype=np.float64)
    w = np.append(d ** -2.1, (tail ** -2.1).sum())
    return float((w * np.arange(1, cap + 1)).sum() / w.sum())


def _distinct(case, n_ids, draws, lo=0.0, hi=1.0):
    """Expected number of distinct ids in [lo n, hi n) among `draws` ids of the case's law."""
    if case.get("ids") != "zipf":
        return n_ids * (hi - lo) * -math.expm1(-draws / n_ids)
    s = case["zipf"]
    edges = np.unique(np.floor(np.logspace(0, math.log10(n_ids + 1.0), 4000)))
    edges = np.clip(edges, 1 + lo * n_ids, 1 + hi * n_ids)
    cdf = (edges ** (1 - s) - 1.0) / ((n_ids + 1.0) ** (1 - s) - 1.0)
    count, mass = np.diff(edges), np.diff(cdf)
    keep = count > 0
    count, mass = count[keep], mass[keep]
    return float((count * -np.expm1(-draws * mass / count)).sum())


def work(case):
    kind = case["kind"]
    if kind in ("affine", "sq", "vq", "hybrid"):
        b = 8 if case["index"] == "int64" else 4
        edges = case["rows"] * _mean_degree(case)
        graph = edges * b + (case["rows"] + 1) * b + 4.0 * case["rows"] * case["dim"]
        if kind == "hybrid":
            hot, cold = (_distinct(case, case["nodes"], edges, *r) for r in ((0.0, case["hot"]), (case["hot"], 1.0)))
            table = hot * (case["dim"] + 4) + cold * (case["codebooks"] + 4) + case["dim"] * (1024 + 8)
        elif kind == "vq":
            table = _distinct(case, case["nodes"], edges) * case["codebooks"] + 1024.0 * case["codebooks"] * case["width"]
        else:
            row = (case["dim"] * case["bits"] + 7) // 8
            table = _distinct(case, case["nodes"], edges) * row + (8 * case["dim"] if kind == "affine" else 20)
        return {"bytes": graph + table, "flops": edges * case["dim"]}
    if kind == "unfused":
        b = 8 if case["index"] == "int64" else 4
        row = -(-case["dim"] // case["width"]) if case["method"] == "vq" else (case["dim"] * case["bits"] + 7) // 8
        edges = case["rows"] * _mean_degree(case)
        return {"bytes": case["sources"] * (8 + row + 4.0 * case["dim"]) + (edges + case["rows"] + 1) * b +
                4.0 * case["rows"] * case["dim"], "flops": edges * case["dim"]}
    if kind == "layer":
        edges = case["dst"] * (1 + case["fanout"]) / 2.0
        n_src = case["dst"] + edges / 2
        books = -(-case["dim"] // case["width"])
        seed_row = case["dim"] * case["seed_bits"] // 8
        return {"bytes": n_src * (8 + books) + case["batch"] * (8 + 4 + seed_row) + (edges + case["dst"]) * 8 +
                1024.0 * books * case["width"] + 8.0 * case["dst"] * case["hidden"] + 16.0 * case["dim"] * case["hidden"],
                "flops": 8.0 * case["dst"] * case["dim"] * case["hidden"] + edges * case["dim"]}
    if kind == "encode_sq":
        values = float(case["nodes"]) * case["dim"]
        return {"bytes": values * 4 + values * case["bits"] / 8 + 8.0 * case["sample"], "flops": values}
    if kind == "train_vq":
        # the rows once (they stay cached), an assignment in every step
        values = float(case["sample"]) * case["dim"]
        return {"bytes": values * 4 + 4.0 * case["dim"] * case["centers"] + 8.0 * case["sample"],
                "flops": case["steps"] * 2.0 * values * case["centers"]}
    if kind == "encode_vq":
        values = float(case["nodes"]) * case["dim"]
        return {"bytes": values * 4 + case["nodes"] * math.ceil(case["dim"] / case["width"]) + 4.0 * case["dim"] * case["centers"],
                "flops": 2.0 * values * case["centers"]}
    return {"bytes": case["rows"] * (4.0 * case["dim"] + 1) + 4.0 * case["dim"] * case["centers"],
            "flops": 2.0 * case["rows"] * case["dim"] * case["centers"]}


def tolerance(case):
    """About four times what another summation order or 64-bit sums change."""
    kind = case["kind"]
    if kind == "affine":
        return {"rel": 2.4e-6, "max": 2e-5}     # min + scale * mean of the codes against the sum of decoded values
    if kind in ("sq", "vq", "hybrid", "unfused"):
        return {"rel": 4e-7, "max": 5e-6}       # fp32 sums over a row's neighbours
    if kind == "layer":
        return {"rel": 1.6e-6, "max": 1e-5}     # fp32 products over the columns, gradients over the rows
    if kind == "encode_sq":
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-5}
    if kind == "train_vq":
        return {"rel": 8e-3, "max": 0.15}       # a row at a near-tie moves its centre, and the steps after it
    return {"differ": 1e-5}                     # a row whose two nearest centres are equal to rounding
