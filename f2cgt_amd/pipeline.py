"""Callers of the operator library, mirrored from the reference's Python with plain tensors in
place of DGL blocks, ShmTensor and torch.distributed (one process, one GPU):

  * the offline encode pipeline: `sq_metadata`, `sq_compress`, `vq_metadata`, `vq_compress`
    (examples/process_compress.py:16-68, 71-144, 147-292), `run` that writes the artefact files
    (`:295-388`) and `load_compress_data` that reads them back (examples/load_dataset.py:63-85);
  * `TensorCache` (examples/tensor_cache.py:36-110): a table of rows on the device or in pinned
    host memory, with an optional device-resident copy of its hottest rows, indexed by global id;
  * `CompressionManager` (examples/compress.py:8-106): keeps the code tables and codebooks,
    serves seed rows (first level) and neighbour rows (second level);
  * `MySAGEConv` (examples/conv.py:9-76): GraphSAGE mean layer whose neighbour aggregation is the
    fused decompress + mean operator.

Everything numerical happens in `F2CGTLib` (f2cgt_amd.load()); this module only moves tensors.
"""
from __future__ import annotations

import math

import numpy as np
import torch
from torch import nn
from torch.nn.modules import module as _modules

import f2cgt_amd


def _capi():
    return f2cgt_amd.load()


# ---- encode pipeline -----------------------------------------------------------------------------
def normalize(data):
    """Every row rescaled to the mean row norm: directions kept, lengths equalised
    (examples/process_compress.py:16-18; same operation order, divide then multiply)."""
    lengths = torch.linalg.vector_norm(data, ord=2, dim=1, keepdim=True)
    return (data / lengths) * lengths.mean()


def sampling(sample_size, num_items, hotness=None, generator=None):
    """Row sample for the codebook statistics (examples/process_compress.py:21-34); with a
    hotness vector the sample follows it, otherwise it is uniform without replacement."""
    if hotness is None:
        return torch.randperm(num_items, generator=generator)[:sample_size]
    p = (hotness.double() / hotness.double().sum()).cpu().numpy()
    p[-1] = 1.0 - p[:-1].sum()
    size = min(sample_size, num_items)
    return torch.from_numpy(np.random.choice(num_items, size, replace=False, p=p))


_PERCENTILES = (0.5, 99.5)


def _percentile_place(n, percent):
    """Where numpy's linear percentile of n float32 values lies: (rank below, rank above, weight of the latter).  numpy
    evaluates the place in the sample's own precision, so (n - 1) * percent / 100 is a float32 here too: beyond 2^24
    values it falls on a whole rank near the exact one."""
    place = np.float32(n - 1) * (np.float32(percent) / np.float32(100))
    if place >= np.float32(n - 1):
        return n - 1, n - 1, np.float32(0)
    below = np.floor(place)
    return int(below), int(below) + 1, np.float32(place - below)


def _between(below, above, weight):
    """The value `weight` of the way from below to above, in float32, from the nearer of the two."""
    with np.errstate(invalid="ignore"):
        gap = above - below
        return below + gap * weight if weight < np.float32(0.5) else above - gap * (np.float32(1) - weight)


def _sq_codebook(lo, hi, level):
    """(fmin, fmax, emin, emax, mean) from the two percentiles and the mean of |x|; the log2 correctly rounded, as on the
    device (torch's float32 log2 is off in the last bit for about 3 values in 10 000)."""
    floor = 1e-5
    fmin, fmax = torch.tensor(max(lo, floor)), torch.tensor(max(hi, 2 * floor))
    level = level + 0.1 if level < 0.1 else level
    emin, emax = (torch.log2(v.double()).float() for v in (fmin, fmax))
    return fmin, fmax, emin, emax + floor, level


def _percentile_places(m, cols, column_slice):
    """Sizes of a full slice and of the last one, and for both the place of either percentile."""
    count = (cols + column_slice - 1) // column_slice
    sizes = [m * min(column_slice, cols), m * (cols - (count - 1) * column_slice)]
    return sizes, [[_percentile_place(n, q) for q in _PERCENTILES] for n in sizes]


def _device_statistics(values, rows, column_slice):
    """Per column slice of float32 GPU rows: (0.5th and 99.5th percentile, mean) of |x|, from exact order statistics
    found on the device; the percentile's interpolation is numpy's, in float32."""
    m = values.shape[0] if rows is None else rows.numel()
    cols = values.shape[1]
    count = (cols + column_slice - 1) // column_slice
    sizes, places = _percentile_places(m, cols, column_slice)
    ranks = [r for per_size in places for place in per_size for r in place[:2]]
    stats = _capi().abs_order_stats(values, rows, column_slice, ranks).cpu().numpy()
    out = []
    for i in range(count):
        last = int(i == count - 1)
        if stats[i, 5] >= 2:
            raise IndexError("a sample id lies outside the table's %d rows" % values.shape[0])
        if stats[i, 5]:
            lo = hi = np.float32("nan")
        else:
            lo, hi = (_between(np.float32(stats[i, 2 * q]), np.float32(stats[i, 2 * q + 1]), places[last][q][2]) for q in (0, 1))
        out.append((lo, hi, torch.tensor(np.float32(stats[i, 4] / sizes[last]))))
    return out


def _device_takes(rows, cols, column_slice):
    """What the device statistics count in: 32 bits of values per slice, 24 of columns, 16 of slices."""
    return (0 < rows * min(cols, column_slice) < 1 << 32 and cols < 1 << 24 and
            (cols + column_slice - 1) // column_slice < 1 << 16)


def sq_metadata(sample):
    """(fmin, fmax, emin, emax, mean) of one column slice from a sample of its rows:
    percentiles of |x| floored at 1e-5 / 2e-5, their log2, mean lifted by 0.1 when
    below 0.1 (examples/process_compress.py:45-68).  A sample on the GPU is reduced there."""
    # (a sample that is part of a graph keeps the host's refusal)
    if sample.is_cuda and sample.numel() and not sample.requires_grad:
        values = sample.float()
        values = values.reshape(-1, values.shape[-1] if values.dim() > 1 else 1)
        if _device_takes(*values.shape, values.shape[1]):
            return _sq_codebook(*_device_statistics(values, None, values.shape[1])[0])
    magnitude = sample.float().abs().cpu()
    # one percentile at a time, as the reference does: numpy returns the sample's own precision for a scalar quantile
    # (float64 for a list of them)
    lo, hi = (np.percentile(magnitude.numpy(), q) for q in _PERCENTILES)
    return _sq_codebook(lo, hi, magnitude.mean())


def _sampled_sq_codebooks(features, sample_index, column_slice):
    """The codebooks from a gathered sample: all slices at once up to 2^28 values (1 GB), else one slice at a time,
    which goes to the host's percentiles where it does not fit the GPU."""
    feat_dim = features.shape[1]
    if sample_index.dim() == 1 and sample_index.numel() * feat_dim <= 1 << 28 and not features.requires_grad:
        try:
            sample = features[sample_index].cuda().float()
            if _device_takes(*sample.shape, column_slice):
                return [_sq_codebook(*values) for values in _device_statistics(sample, None, column_slice)]
        except torch.OutOfMemoryError:
            pass
    per_slice = []
    for lo in range(0, feat_dim, column_slice):
        sample = features[sample_index, lo:lo + column_slice]
        try:
            per_slice.append(sq_metadata(sample.cuda()))
        except torch.OutOfMemoryError:
            if sample.is_cuda:
                raise
            per_slice.append(sq_metadata(sample))
    return per_slice


def _bad_rows(stats):
    """Whether an id of the sample that statistics were made of lies outside its table."""
    pending = getattr(stats, "bad_rows", None)
    return pending.wait() if pending is not None else stats.cpu().numpy()[:, 5].max() >= 2


def sq_compress(features, target_bits, column_slice, hotness=None, sample_index=None, batch_rows=1_000_000):
    """-> (storage, codebooks).  storage: int8 [N, ceil(D * bits / 8)] holding the packed bit
    patterns (bits <= 8) or int16 [N, D]; codebooks fp32 [ceil(D / column_slice), 5] on the GPU
    (examples/process_compress.py:71-144, single process)."""
    capi = _capi()
    num_items, feat_dim = features.shape
    if sample_index is None:
        sample_index = sampling(250_000, num_items, hotness)
    sample_index = sample_index.to(features.device)
    stats = None
    if (features.is_cuda and features.dtype == torch.float32 and features.stride(1) == 1 and features.stride(0) >= feat_dim and
            sample_index.dtype == torch.int64 and sample_index.dim() == 1 and not features.requires_grad and
            _device_takes(sample_index.numel(), feat_dim, column_slice)):
        # the sample's rows are read in place, the codebooks made where they are used; the ids' check comes to the host
        # from the first of these kernels, so that only that one is waited for
        places = _percentile_places(sample_index.numel(), feat_dim, column_slice)[1]
        codebooks, stats = capi.sq_codebooks(features, sample_index, column_slice,
                                             [r for per_size in places for place in per_size for r in place[:2]],
                                             [place[2] for per_size in places for place in per_size])
        codebooks = codebooks.cuda()      # (the codes are made on the current device, wherever the table lies)
    else:
        per_slice = [[float(v) for v in values] for values in _sampled_sq_codebooks(features, sample_index, column_slice)]
        codebooks = (torch.tensor(per_slice, dtype=torch.float32) if per_slice else torch.zeros((0, 5))).cuda()
    if target_bits <= 8:
        dtype, tdim = torch.int8, int(math.ceil(feat_dim / 8 * target_bits))
    elif target_bits <= 16:
        dtype, tdim = torch.int16, feat_dim
    else:
        raise NotImplementedError
    out = torch.empty((num_items, tdim), dtype=dtype, device="cuda")
    for start in range(0, num_items, batch_rows):
        end = min(start + batch_rows, num_items)
        data = features[start:end].cuda().to(torch.float32)
        # one pass; the reference calls sq_compress, casts and packs (process_compress.py:128-139)
        capi.sq_encode(data, codebooks, target_bits, column_slice, out[start:end])
    if stats is not None and _bad_rows(stats):
        raise IndexError("a sample id lies outside the table's %d rows" % num_items)
    return out, codebooks


def _circle_centers(n, width, generator=None, slices=1):
    """[slices * n, width] random unit-circle pairs on the host, the draws of one slice after those of the one before."""
    half = width // 2
    if width % 2 == 0:
        angles = torch.rand((slices * n, half), generator=generator) * (2 * math.pi)
        return torch.cat([torch.cos(angles), torch.sin(angles)], dim=1).float()
    parts = []
    for _ in range(slices):
        radii = torch.rand((n, 1), generator=generator)
        angles = torch.rand((n, half + 1), generator=generator) * (2 * math.pi)
        parts.append(radii * torch.cat([torch.cos(angles[:, :half]), torch.sin(angles)], dim=1))
    return torch.cat(parts).float()


class KMeansTrainer:
    """Codebook trainer of the offline compressor (examples/my_kmeans.py:73-113, 150-184), on the
    device from start to finish: assignment by `kmeans_predict`, centre update and stopping rule by
    `kmeans_update`.

    As in the reference: `cosine` starts from random unit-circle pairs (cos / sin of uniform angles,
    :9-24), `euclidean` from distinct random non-zero rows (:27-31); a centre is the plain mean of its
    members whatever the metric and keeps its value when it has none (:128-147); the fit ends when
    (sum_c |centre shift|)^2 < tol, with tol growing by a factor 1.2 per iteration (:100-111).
    The rule is evaluated by the update kernel, which freezes the centres when it holds; the host
    reads the flag every `check_every` iterations, so the loop runs without a read-back per step.
    """

    def __init__(self, num_clusters, metric="cosine", tol=1e-4, mode="fast", max_iter=1000, check_every=8,
                 generator=None):
        if metric not in ("cosine", "euclidean"):
            raise ValueError("metric must be 'cosine' or 'euclidean'")
        if mode not in ("fast", "normal"):
            raise ValueError("mode must be 'fast' or 'normal'")
        self.num_clusters, self.metric, self.tol, self.mode = num_clusters, metric, tol, mode
        self.max_iter, self.check_every, self.generator = max_iter, check_every, generator
        self.centers, self.n_iter = None, 0

    def _initial_centers(self, data):
        n, width = self.num_clusters, data.shape[1]
        if self.metric == "cosine":
            return _circle_centers(n, width, self.generator).cuda()
        alive = torch.nonzero(torch.count_nonzero(data, dim=1)).flatten()
        if alive.numel() < n:
            raise ValueError("fewer non-zero rows than clusters")
        pick = torch.randperm(alive.numel(), generator=self.generator)[:n].to(alive.device)
        return data[alive[pick]].float().cuda()

    def fit(self, data):
        capi = _capi()
        data = data.float().cuda().contiguous()
        centers = self._initial_centers(data).contiguous()
        metric = "cosine" if self.metric == "cosine" else "l2"
        stop = torch.zeros((1,), dtype=torch.int32, device="cuda")
        tol, self.n_iter = float(self.tol), 0
        for it in range(self.max_iter):
            labels = capi.kmeans_predict(data, centers, metric)
            capi.kmeans_update(data, labels, centers, stop, 2, tol)
            tol *= 1.2
            self.n_iter += 1
            if it % self.check_every == self.check_every - 1 and int(stop.item()):
                break
        if int(stop.item()) == 2:
            # the centre shift is not a number (NaN or infinite input): the reference's trainer gives
            # up on such a fit (examples/my_kmeans.py:108-109); so does this one, loudly
            import warnings
            warnings.warn("KMeansTrainer.fit: the centre shift became NaN; no centres were produced")
            self.centers = None
            return
        self.centers = centers

    def get_centers(self):
        return self.centers

    def predict(self, data, normalize_weights=False):
        metric = "cosine" if self.metric == "cosine" else "l2"
        return _capi().kmeans_predict(data.float().cuda().contiguous(), self.centers, metric)


def _rim_quantile(width):
    return min(1.0, 0.00625 * (width / 8))


def _rim_place(m, width):
    """Where torch's linear quantile of m float32 values lies: (rank below, rank above, weight of the latter), in the
    values' own precision."""
    place = np.float32(_rim_quantile(width)) * np.float32(m - 1)
    below = np.floor(place)
    return int(below), int(np.ceil(place)), float(np.float32(place - below))


def _train_all_slices(features, n_clusters, column_slice, sample_index, max_iter):
    """The codebooks of vq_metadata with every step made for all slices at once, or None where that is not covered: more
    slices, centres or columns than a step takes, samples that are no plain list of row ids, empty or beyond 2^24 rows
    (torch's quantile) or 2^28 values."""
    capi = _capi()
    feat_dim = features.shape[1]
    slices = (feat_dim + column_slice - 1) // column_slice
    m = sample_index.numel()
    if not (sample_index.dtype == torch.int64 and sample_index.dim() == 1 and 0 < m <= 1 << 24 and m * feat_dim <= 1 << 28 and
            capi.kmeans_slices_covers(slices, n_clusters, column_slice) and features.shape[0] > 0):
        return None
    if (features.is_cuda and features.device.index == torch.cuda.current_device() and features.dtype == torch.float32 and
            features.stride(1) == 1 and features.stride(0) >= feat_dim):
        table, rows = features, sample_index.to(features.device)
    else:
        table, rows = features[sample_index.to(features.device)].to(torch.float32).cuda(), None
    data, lengths, bad_row = capi.slice_rows(table, rows, column_slice)
    last = feat_dim - (slices - 1) * column_slice
    places = [_rim_place(m, width) for width in (min(column_slice, feat_dim), last)]
    stats = capi.abs_order_stats(lengths, None, 1, [r for p in places for r in (p[0], p[1], p[0], p[1])])
    keep = capi.keep_rows(lengths, stats, places[0][2], places[1][2])
    # the draws of the trainers, slice after slice
    whole = slices - 1 if last < column_slice else slices
    start = torch.zeros((slices, n_clusters, column_slice))
    if whole:
        start[:whole] = _circle_centers(n_clusters, column_slice, slices=whole).view(whole, n_clusters, column_slice)
    if whole < slices:
        start[whole, :, :last] = _circle_centers(n_clusters, last)
    centers = start.cuda()
    flags, codebooks = capi.kmeans_slices_fit(data, keep, centers, "cosine", 2, 5e-2, 1.2, max_iter, 8, bad_row, True)
    *stop, bad, nan = flags.tolist()
    if rows is not None and bad:
        raise IndexError("a sample id lies outside the table's %d rows" % features.shape[0])
    worst = max(stop)
    if worst == 3:       # their quantile is no number: a NaN among the lengths, or infinities
        raise RuntimeError("a column slice has no rows to train on")
    if worst == 2:
        import warnings
        warnings.warn("vq_metadata: the centre shift became NaN; no centres were produced")
        raise TypeError("a column slice has no centres")
    if nan:
        raise ValueError("codebooks has nan")
    return codebooks


def vq_metadata(features, n_clusters, column_slice, hotness=None, sample_index=None, max_iter=1000):
    """Codebooks fp32 [ceil(D / column_slice), n_clusters, column_slice]: per slice, rows of a
    sample inside the rim quantile are dropped, k-means (cosine, tol 5e-2) runs on the rest and the
    centres are rescaled to their mean norm (examples/process_compress.py:147-182)."""
    capi = _capi()
    num_items, feat_dim = features.shape
    if sample_index is None:
        sample_index = sampling(150_000, num_items, hotness)
    num_slice = (feat_dim + column_slice - 1) // column_slice
    draws = torch.get_rng_state()
    try:
        codebooks = _train_all_slices(features, n_clusters, column_slice, sample_index, max_iter)
    except torch.OutOfMemoryError:        # no room for the sample's slices side by side: one at a time, with the same draws
        codebooks = None
        torch.set_rng_state(draws)
    if codebooks is None:
        codebooks = torch.zeros((num_slice, n_clusters, column_slice), device="cuda", dtype=torch.float32)
        per_slice = range(num_slice)
    else:
        per_slice = ()
    for i in per_slice:
        lo, hi = i * column_slice, min((i + 1) * column_slice, feat_dim)
        data = features[sample_index.to(features.device), lo:hi].to(torch.float32).cuda()
        distance = data.norm(dim=1, p=2)
        rim = torch.quantile(distance, _rim_quantile(data.shape[1]))
        data = data[torch.ge(distance, rim)].contiguous()
        km = KMeansTrainer(n_clusters, metric="cosine", tol=5e-2, max_iter=max_iter)
        km.fit(data)
        centers = normalize(km.get_centers())
        codebooks[i, :, :hi - lo] = centers
    if per_slice and torch.isnan(codebooks).any():
        raise ValueError("codebooks has nan")
    return codebooks


def vq_compress(features, n_clusters, column_slice, hotness=None, codebooks=None, sample_index=None,
                batch_rows=1_000_000):
    """-> (codes, codebooks).  codes: uint8 (K <= 256) or int16 [N, n_slices], one nearest
    (cosine) centre per column slice (examples/process_compress.py:185-292, single process)."""
    capi = _capi()
    num_items, feat_dim = features.shape
    if codebooks is None:
        codebooks = vq_metadata(features, n_clusters, column_slice, hotness, sample_index)
    num_slice = codebooks.shape[0]
    if n_clusters <= 256:
        dtype = torch.uint8
    elif n_clusters <= 32767:
        dtype = torch.int16
    else:
        raise NotImplementedError("more than 32767 centres do not fit the int16 code type")
    out = torch.empty((num_items, num_slice), dtype=dtype, device="cuda")
    predictors = None
    for start in range(0, num_items, batch_rows):
        end = min(start + batch_rows, num_items)
        # float32 rows on the device and up to 256 centres: all slices in one launch, the rows read in place
        if (tuple(codebooks.shape[2:]) == (column_slice,) and
                capi.vq_encode_slices(features[start:end], codebooks, out[start:end], "cosine")):
            continue
        if predictors is None:
            predictors = [capi.KMeans(codebooks[i].contiguous(), "cosine") for i in range(num_slice)]
        for i in range(num_slice):
            lo, hi = i * column_slice, min((i + 1) * column_slice, feat_dim)
            if hi <= lo:
                continue
            data = torch.zeros((end - start, column_slice), device="cuda", dtype=torch.float32)
            data[:, :hi - lo] = features[start:end, lo:hi].to(torch.float32)
            labels = predictors[i].predict(data, normalize_weights=False)
            out[start:end, i] = labels.to(dtype)
    return out, codebooks


def run(root, features, seeds=None, hotness=None, target_compression_ratio=32, n_clusters=256):
    """Compresses a feature table and writes the artefacts the training scripts load
    (examples/process_compress.py:295-388, single process, column slices as for one rank):

      * `compression_meta.pt`: dict with `methods` (['sq'] / ['vq'], preceded by 'sq' when seed
        rows get their own table), `codebooks` (CPU tensors, one per level), `configs`
        ((column_slice, target_bits) per level, target_bits -1 for VQ), `feat_dim`, `data`
        (name -> (dtype, shape) of each code table) and `seeds` (ids of the seed rows);
      * `compression_data.pt`: the code table of every row;
      * `seeds_compression_data.pt`: the code table of the seed rows (SQ at one eighth of the
        element width in bits, i.e. 4-bit codes for fp32 features).

    A ratio up to the element width in bits selects SQ with `width / ratio` bits per value; a
    larger one selects VQ with `ratio / element_size` columns per code byte (twice that for
    more than 256 centres).  Returns the meta dict."""
    import os
    feat_dim = features.shape[1]
    width_bits = features.element_size() * 8
    methods, configs, codebook_list, data, meta = [], [], [], {}, {}
    slice_of_row = (feat_dim + 7) // 8 * 8
    if seeds is not None:
        seed_bits = width_bits // 8
        seed_rows = features[seeds.to(features.device)]
        seed_codes, seed_cbs = sq_compress(seed_rows, seed_bits, slice_of_row, None)
        methods.append("sq")
        configs.append((slice_of_row, seed_bits))
        codebook_list.append(seed_cbs.cpu())
        data["seeds_compression_data"] = (seed_codes.dtype, seed_codes.shape)
        meta["seeds"] = seeds.cpu()
        torch.save(seed_codes.cpu(), os.path.join(root, "seeds_compression_data.pt"))
        del seed_codes
    if target_compression_ratio <= width_bits:
        target_bits = int(width_bits / target_compression_ratio)
        codes, cbs = sq_compress(features, target_bits, slice_of_row, hotness)
        methods.append("sq")
        configs.append((slice_of_row, target_bits))
    else:
        column_slice = target_compression_ratio // features.element_size()
        if n_clusters > 256:
            column_slice *= 2
        codes, cbs = vq_compress(features, n_clusters, column_slice, hotness)
        methods.append("vq")
        configs.append((column_slice, -1))
    codebook_list.append(cbs.cpu())
    data["compression_data"] = (codes.dtype, codes.shape)
    meta.update(methods=methods, codebooks=codebook_list, configs=configs, feat_dim=feat_dim, data=data)
    torch.save(meta, os.path.join(root, "compression_meta.pt"))
    torch.save(codes.cpu(), os.path.join(root, "compression_data.pt"))
    return meta


def load_compress_data(root):
    """The dict `CompressionManager` takes, read back from the files `run` wrote: the meta dict
    with every code table named in `data` added under its name
    (examples/load_dataset.py:63-85 without the shared-memory staging)."""
    import os
    meta = torch.load(os.path.join(root, "compression_meta.pt"), weights_only=True)
    for name, (dtype, shape) in meta["data"].items():
        table = torch.load(os.path.join(root, name + ".pt"), weights_only=True)
        if table.dtype != dtype or tuple(table.shape) != tuple(shape):
            raise ValueError("%s.pt does not match its entry in compression_meta.pt" % name)
        meta[name] = table
    return meta


# ---- runtime callers -------------------------------------------------------------------------------
class TensorCache:
    """examples/tensor_cache.py:36-110 without ShmTensor.

    `data` is a 2-D table of rows (code rows or plain features).  A host table is copied once
    into pinned memory that the device can address (the reference pins the shared-memory table in
    place; registering existing memory is not available here), and `cache[index]` reads its rows
    over the host link; `create_cache(capacity, hotness)` moves the whole table to the device
    when it fits in `capacity` bytes and otherwise keeps a device copy of the hottest rows plus a
    dense int32 array id -> cache slot (-1 = not cached) where the reference keeps a GPU hash
    map.  The array costs 4 bytes per table row and is charged to the capacity.
    `index` is a device tensor of int32/int64 ids; the result is a new device tensor."""

    def __init__(self, data):
        if data.dim() != 2:
            raise ValueError("TensorCache holds a 2-D table of rows")
        if data.device.type == "cpu":
            pinned = torch.empty(data.shape, dtype=data.dtype, pin_memory=True)
            pinned.copy_(data)
            data = pinned
        self.data = data.contiguous()
        self.gpu_data = None
        self.slot_map = None
        self.has_cache = False

    def __getitem__(self, index):
        capi = _capi()
        if index.dtype not in (torch.int32, torch.int64):
            index = index.long()
        if self.has_cache:
            return capi.fetch_rows(self.data, index, self.gpu_data, self.slot_map)
        return capi.fetch_rows(self.data, index)

    def create_cache(self, cache_capacity, hotness):
        if cache_capacity <= 0:
            return
        full_size = self.data.numel() * self.data.element_size()
        if full_size <= cache_capacity:
            self.data = self.data.cuda()
            return
        row_bytes = self.data.shape[1] * self.data.element_size()
        cache_num = int((cache_capacity - 4 * self.data.shape[0]) // row_bytes)
        if cache_num <= 0:
            return
        _, candidates = torch.sort(hotness, descending=True)
        candidates = candidates[:cache_num]
        self.gpu_data = self.data[candidates.to(self.data.device)].cuda()
        self.slot_map = torch.full((self.data.shape[0],), -1, dtype=torch.int32, device="cuda")
        self.slot_map[candidates.cuda().long()] = torch.arange(candidates.numel(), dtype=torch.int32, device="cuda")
        self.has_cache = True

    def clear_cache(self):
        self.has_cache = False
        self.gpu_data = None
        self.slot_map = None

    def compute_weight_size(self, hotness):
        """(bytes of the whole table, bytes of a row weighted by the mean hotness of the rows that are
        ever touched): the two inputs of the reference's cache-split cost model
        (examples/tensor_cache.py:102-106)."""
        row_bytes = self.data.shape[1] * self.data.element_size()
        touched = hotness[hotness > 0]
        return self.data.shape[0] * row_bytes, row_bytes * float(touched.float().mean())


class CompressionManager:
    """examples/compress.py:8-106 on plain tensors.

    `compress_data` keys (the layout of the reference's `compression_meta.pt` + data tensors):
    `methods` (list of 'sq' / 'vq', one entry, or two for seeds + everything), `feat_dim`,
    `configs` (per level (column_slice, target_bits)), `codebooks` (per level), `compression_data`
    (code table of the last level, [N, src_dim]), and for two levels `seeds_compression_data`
    (code table of the seed rows) with `seeds` (their global ids).

    The code tables sit behind `TensorCache`.  `device_resident=True` (the default: the largest
    table of the benchmark configurations is 5.76 GB against 288 GB of device memory) moves them
    to the device at construction, the reference's whole-table cache
    (examples/tensor_cache.py:66-70); `False` leaves host tables in pinned host memory until
    `manager.data.create_cache(capacity, hotness)` is called, as the reference does.
    """

    def __init__(self, compress_data, fusion=False, device_resident=True):
        self.meta = compress_data
        self.methods = compress_data["methods"]
        self.feat_dim = compress_data["feat_dim"]
        self.configs = compress_data["configs"]
        self.codebooks = [c.cuda() for c in compress_data["codebooks"]]
        place = (lambda t: t.cuda()) if device_resident else (lambda t: t)
        self.data = TensorCache(place(compress_data["compression_data"]))
        self.seeds_data = None
        self.is_two_level = len(self.methods) >= 2
        self.is_fusion = fusion
        # the seed rows are fetched and decoded on a stream of their own while the caller goes on to
        # sample and gather the block (examples/compress.py:36-53); default priority
        self.seeds_task_stream = torch.cuda.Stream()
        self.seeds_task_event = torch.cuda.Event()
        self.check_seed_keys = True   # a host round trip per call; the reference's hash map query has no such check
        if self.is_two_level:
            self.seeds_data = TensorCache(place(compress_data["seeds_compression_data"]))
            keys = compress_data["seeds"].long().cuda()
            # global id -> row of the seed table (the reference keeps a GPU hash map)
            self.seed_slot = torch.full((self.data.data.shape[0],), -1, dtype=torch.int32, device="cuda")
            self.seed_slot[keys] = torch.arange(keys.numel(), dtype=torch.int32, device="cuda")

    def _decompress(self, level, data):
        capi = _capi()
        if self.methods[level] == "vq":
            return capi.vq_decompress(data, self.codebooks[level], self.feat_dim)
        return capi.sq_decompress(data, self.codebooks[level], self.configs[level][1], self.configs[level][0],
                                  self.feat_dim)

    def _decode_rows(self, level, cache, keys):
        """Decoded rows `keys` of a code table: read by the decoder itself where the whole table is in device memory,
        fetched and decoded otherwise."""
        if not cache.data.is_cuda or cache.has_cache:
            return self._decompress(level, cache[keys])
        capi = _capi()
        if keys.dtype not in (torch.int32, torch.int64):
            keys = keys.long()
        if self.methods[level] == "vq":
            return capi.vq_decompress_rows(cache.data, keys, self.codebooks[level], self.feat_dim)
        return capi.sq_decompress_rows(cache.data, keys, self.codebooks[level], self.configs[level][1],
                                       self.configs[level][0], self.feat_dim)

    def get_seeds_data(self, seeds_key):
        """Decoded first-level rows of `seeds_key`; the result may be used on another stream only after
        `seeds_task_event` (reorganize_seeds_data waits for it).  Produced on `seeds_task_stream`, or, where the one kernel
        that looks the rows up, checks, fetches and decodes them is followed by a wait for its check, on the current stream:
        the call returns with the rows made either way, and handing the work to another stream and back took longer than
        the kernel (57 -> 25 us of the host's time a minibatch)."""
        if not self.is_two_level:
            return None
        seeds = self.seeds_data
        in_one = (self.methods[0] == "sq" and seeds.data.is_cuda and not seeds.has_cache and
                  seeds_key.dtype in (torch.int32, torch.int64))
        if in_one and self.check_seed_keys and seeds_key.is_cuda:     # (keys on the host are refused below)
            seeds_feature = self._decode_seeds(seeds_key)
            self.seeds_task_event.record()
            return seeds_feature
        side = self.seeds_task_stream
        side.wait_stream(torch.cuda.current_stream())      # seeds_key may still be in the making
        with torch.cuda.stream(side):
            # the caller may drop seeds_key as soon as this returns: tie its memory to the side stream
            seeds_key.record_stream(side)
            if in_one:
                seeds_feature = self._decode_seeds(seeds_key)
                self.seeds_task_event.record(side)
                return seeds_feature
            slots = self.seed_slot[seeds_key.long()].long()
            if self.check_seed_keys and bool((slots < 0).any()):
                raise KeyError("a requested id is not a seed row")
            seeds_feature = self._decompress(0, self.seeds_data[slots])
            self.seeds_task_event.record(side)
        return seeds_feature

    def _decode_seeds(self, seeds_key):
        return _capi().sq_decompress_rows(self.seeds_data.data, seeds_key, self.codebooks[0], self.configs[0][1],
                                          self.configs[0][0], self.feat_dim, self.seed_slot, self.check_seed_keys)

    def get_all_data(self, keys):
        if self.is_fusion:
            return self.data[keys]
        return self._decode_rows(1 if self.is_two_level else 0, self.data, keys)

    def aggregate_global(self, indptr, indices, input_nodes):
        """Mean aggregation of a sampled block straight from the device-resident code table:
        `indices` are positions in `input_nodes` (the block's source ids), which are composed
        into global ids so that the fused operator reads the table rows itself and the gathered
        copy of `get_all_data` is never written.  Same result as
        `fused_op(get_all_data(input_nodes), ..., indptr, indices)`."""
        if not self.data.data.is_cuda:
            raise RuntimeError("aggregate_global needs the code table on the device")
        capi = _capi()
        level = 1 if self.is_two_level else 0
        global_ids = input_nodes.to(indices.dtype)[indices.long()]
        if self.methods[level] == "vq":
            return capi.vq_decompress_spmm_csr(self.data.data, self.codebooks[level], indptr, global_ids,
                                               self.feat_dim)
        return capi.sq_decompress_spmm_csr(self.data.data, self.codebooks[level], indptr, global_ids,
                                           self.configs[level][1], self.configs[level][0], self.feat_dim)

    def reorganize_seeds_data(self, seeds_feature, all_feature, num_dst):
        if seeds_feature is not None:
            # the consumer joins the seed stream here (examples/compress.py:74-75)
            current = torch.cuda.current_stream()
            current.wait_event(self.seeds_task_event)
            seeds_feature.record_stream(current)
        if not self.is_fusion:
            if seeds_feature is None:
                return None
            num_seeds = seeds_feature.shape[0]
            return torch.cat([seeds_feature, all_feature[num_seeds:num_dst]], dim=0)
        if self.is_two_level:
            num_seeds = seeds_feature.shape[0]
            part = all_feature[num_seeds:num_dst]
        else:
            part = all_feature[:num_dst]
        part_feature = self._decompress(1 if self.is_two_level else 0, part.contiguous())
        if self.is_two_level:
            return torch.cat([seeds_feature, part_feature], dim=0)
        return part_feature


_MODULE_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def _plain_linear(layer):
    """Whether calling `layer` is nn.Linear's own product and nothing else: no subclass or replaced forward, no
    parametrization (which is a subclass), no hook on it or on all modules."""
    return (type(layer) is nn.Linear and "forward" not in layer.__dict__ and
            not any(getattr(layer, name) for name in _MODULE_HOOKS) and
            not any(getattr(_modules, "_global" + name) for name in _MODULE_HOOKS))


class MySAGEConv(nn.Module):
    """examples/conv.py:9-76.  `forward(csc, feat)`: `csc = (indptr, indices)` of the block
    (destination rows x source rows), `feat = (h_self, h_neigh)`; with a fusing manager `h_neigh`
    is the compressed code rows of the source nodes and the aggregation decodes them on the fly.

    The two products, their sum, the bias and a ReLU are one call (`sage_linear`) where the two layers are plain
    `nn.Linear`s on dense fp32 device tensors and the inputs are not differentiated; the layers' own operators otherwise,
    also under transforms, modes, autocast and tracing.  The values are the operators' own, and so is the ReLU's mask: a
    kernel makes them at the sizes at which it adds in the library's order (a minibatch's, up to 128 columns), the
    library's products at all others.  The gradients are one or two launches up to 4096 rows, beyond which the
    pass is the operators'.  A step at 1024 x (128 + 128) -> 256 takes the host 65 us where the operators take 187, the
    device 23 where they take 44."""

    def __init__(self, in_feats, out_feats, aggregator_type, compression_manager, bias=True, norm=None,
                 activation=None):
        super().__init__()
        if aggregator_type != "mean":
            raise ValueError("the fused layer aggregates by mean only (got %r)" % (aggregator_type,))
        src_width, dst_width = (in_feats, in_feats) if isinstance(in_feats, int) else tuple(in_feats)
        self.sm = compression_manager
        self.activation, self.norm = activation, norm
        # the reference's attribute names (examples/conv.py:29-31): checkpoints of either load into the other
        self.fc_neigh = nn.Linear(src_width, out_feats, bias=False)
        self.fc_self = nn.Linear(dst_width, out_feats, bias=bias)
        self.reset_parameters()

    def reset_parameters(self):
        """Glorot-uniform weights scaled for a ReLU that follows (examples/conv.py:38-42)."""
        for layer in (self.fc_self, self.fc_neigh):
            nn.init.xavier_uniform_(layer.weight, gain=nn.init.calculate_gain("relu"))

    def forward(self, csc, feat):
        capi = _capi()
        indptr, indices = csc
        h_self, h_neigh = feat
        num_dst = indptr.numel() - 1
        if h_self is None:
            h_self = h_neigh[:num_dst]
        sm = self.sm
        if sm is None or not sm.is_fusion:
            h_neigh = capi.spmm_csr(h_neigh, indptr, indices)
        else:
            level = 1 if sm.is_two_level else 0
            if sm.methods[level] == "vq":
                h_neigh = capi.vq_decompress_spmm_csr(h_neigh, sm.codebooks[level], indptr, indices, sm.feat_dim)
            else:
                h_neigh = capi.sq_decompress_spmm_csr(h_neigh, sm.codebooks[level], indptr, indices,
                                                      sm.configs[level][1], sm.configs[level][0], sm.feat_dim)
        relu = self.activation is torch.relu or self.activation is nn.functional.relu
        rst = None
        if _plain_linear(self.fc_self) and _plain_linear(self.fc_neigh) and self.fc_neigh.bias is None:
            rst = capi.sage_linear(h_self, h_neigh, self.fc_self.weight, self.fc_neigh.weight, self.fc_self.bias, relu)
        if rst is None:
            rst, relu = self.fc_self(h_self) + self.fc_neigh(h_neigh), False
        if self.activation is not None and not relu:
            rst = self.activation(rst)
        if self.norm is not None:
            rst = self.norm(rst)
        return rst
