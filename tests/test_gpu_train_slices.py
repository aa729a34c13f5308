"""Codebook training with every step made for all column slices at once: the slices of a sample, the rows that take part,
one Lloyd step against float64, and the trained codebooks against the slice-by-slice path."""
import numpy as np
import pytest
import torch

import f2cgt_amd
from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


# widths with one to sixteen lanes per row, last slices of one column and of all, rows that start at any float
@pytest.mark.parametrize("m,n_rows,dim,k,start,pitch", [
    (1, 1, 1, 1, 0, 1), (70, 50, 17, 4, 1, 19), (300, 1000, 96, 16, 0, 96), (257, 300, 45, 7, 3, 45), (130, 200, 100, 32, 2, 101),
    (64, 64, 61, 60, 0, 64), (1000, 500, 5, 64, 0, 5)])
def test_slice_rows(m, n_rows, dim, k, start, pitch):
    print("case slice_rows", m, n_rows, dim, k, start, pitch, flush=True)
    g = torch.Generator().manual_seed(m + dim)
    flat = torch.zeros(n_rows * pitch + start, device="cuda")
    x = flat[start:].view(n_rows, pitch)[:, :dim]
    x.copy_(torch.randn((n_rows, dim), generator=g))
    rows = torch.randint(-n_rows, n_rows, (m,), generator=g)
    slices = (dim + k - 1) // k
    out, norms, bad = f2cgt_amd.load().slice_rows(x, rows.cuda(), k)
    want = torch.zeros((m, slices * k))
    want[:, :dim] = x.cpu()[rows]
    want = want.view(m, slices, k).transpose(0, 1)
    assert torch.equal(out.cpu(), want) and int(bad.item()) == 0
    # a sum of up to 64 squares and a root: below 2^-19 of the length
    assert torch.allclose(norms.cpu().double(), want.double().norm(dim=2).t(), rtol=2e-6, atol=0)
    rows[m // 2] = n_rows
    assert int(f2cgt_amd.load().slice_rows(x, rows.cuda(), k)[2].item()) == 1


@pytest.mark.parametrize("m", [1, 2, 31, 32, 33, 64, 65, 1000, 70001])
@pytest.mark.parametrize("width,last", [(16, 16), (8, 3), (64, 1)])
def test_keep_rows(m, width, last):
    print("case keep_rows", m, width, last, flush=True)
    lib = f2cgt_amd.load()
    g = torch.Generator().manual_seed(m)
    norms = torch.rand((m, 3), generator=g).round(decimals=3).cuda()        # with equal lengths among them
    places = [pipeline._rim_place(m, w) for w in (width, last)]
    stats = lib.abs_order_stats(norms, None, 1, [r for p in places for r in (p[0], p[1], p[0], p[1])])
    keep = lib.keep_rows(norms, stats, places[0][2], places[1][2]).cpu().numpy().view(np.uint32)
    bits = np.unpackbits(keep.view(np.uint8), axis=1, bitorder="little")
    assert not bits[:, m:].any()
    for s in range(3):
        rim = torch.quantile(norms[:, s], pipeline._rim_quantile(last if s == 2 else width))
        assert np.array_equal(bits[s, :m].astype(bool), torch.ge(norms[:, s], rim).cpu().numpy())
    norms[m - 1, 1] = float("nan")
    stats = lib.abs_order_stats(norms, None, 1, [r for p in places for r in (p[0], p[1], p[0], p[1])])
    assert not lib.keep_rows(norms, stats, places[0][2], places[1][2])[1].any()


def step64(x, keep, centers, metric, values=None):
    """One Lloyd step of a slice in float64: the means of the rows, or of `values` in their places, by label."""
    x, c = x.astype(np.float64), centers.astype(np.float64)
    values = x if values is None else values.astype(np.float64)
    if metric == "cosine":
        d = 1.0 - (x @ c.T) / np.maximum(np.linalg.norm(x, axis=1)[:, None] * np.linalg.norm(c, axis=1)[None], 1e-8)
    else:
        d = ((x[:, None] - c[None]) ** 2).sum(-1)
    label = d.argmin(1)
    new = c.copy()
    for j in range(c.shape[0]):
        mine = keep & (label == j)
        if mine.any():
            new[j] = values[mine].mean(0)
    return new


# n and k: every operand step, one tile and several, chunks that end in padding; m: fewer groups than workgroups and more
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("slices,m,n,k,masked", [
    (1, 1, 1, 4, False), (3, 31, 5, 3, True), (6, 5000, 256, 16, True), (2, 33, 32, 17, False), (5, 700, 33, 8, True),
    (1, 20000, 64, 32, True), (2, 900, 100, 40, True), (1, 400, 40, 64, False), (200, 64, 16, 8, True), (7, 3000, 130, 15, False)])
def test_one_step(metric, slices, m, n, k, masked):
    print("case kmeans_slices", metric, slices, m, n, k, masked, flush=True)
    rng = np.random.default_rng(m + n + k)
    x = rng.standard_normal((slices, m, k)).astype(np.float32)
    c = rng.standard_normal((slices, n, k)).astype(np.float32)
    keep = rng.random((slices, m)) < 0.7 if masked else np.ones((slices, m), bool)
    bits = None
    if masked:
        padded = np.zeros((slices, (m + 31) // 32 * 32), bool)
        padded[:, :m] = keep
        bits = torch.from_numpy(np.packbits(padded, axis=1, bitorder="little").view(np.int32).copy()).cuda()
    lib = f2cgt_amd.load()
    assert lib.kmeans_slices_covers(slices, n, k)
    centers = torch.from_numpy(c).cuda()
    flags = lib.kmeans_slices_fit(torch.from_numpy(x).cuda(), bits, centers, metric, 0, 0.0, 1.0, 1, 8)
    got = centers.cpu().numpy().astype(np.float64)
    assert flags.tolist() == [0] * slices
    for s in range(slices):
        want = step64(x[s], keep[s], c[s], metric)
        # each set's fp64 sums are rounded once, which makes 2^-24 of the mean of |x| at most, their total and its
        # quotient once more each
        bound = 1.01 * 2.0 ** -24 * (step64(x[s], keep[s], c[s], metric, np.abs(x[s])) + 2 * np.abs(want))
        assert (np.abs(got[s] - want) <= bound).all()


@pytest.mark.parametrize("metric", ["cosine", "l2"])
def test_sums_hold_more_than_fp32(metric):
    """Rows of one value that an fp32 sum beyond 256 rounds down every time: 2^-24 100 of the mean and more, where each of a
    workgroup's sums has some 600 rows."""
    value = 1.0 + 0.4 * 2.0 ** -15
    x = torch.full((1, 300_000, 5), value)
    x[:, ::2] *= -1.0
    centers = torch.tensor([[[1.0] * 5, [-1.0] * 5]]).cuda()
    f2cgt_amd.load().kmeans_slices_fit(x.cuda(), None, centers, metric, 0, 0.0, 1.0, 1, 8)
    want = float(np.float32(value))
    got = centers.cpu().double()[0]
    assert (got[0] - want).abs().max() <= 3.03 * 2.0 ** -24 * want and (got[1] + want).abs().max() <= 3.03 * 2.0 ** -24 * want


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("scale", [1e21, 1e30])
@pytest.mark.parametrize("k", [16, 30])
def test_one_step_with_centres_whose_squares_overflow(metric, scale, k):
    print("case kmeans_slices overflow", metric, scale, k, flush=True)
    rng = np.random.default_rng(k)
    x, c = rng.standard_normal((2, 700, k)), rng.standard_normal((2, 40, k))
    x[:, ::2] *= scale
    c[:, ::3] *= scale
    x, c = x.astype(np.float32), c.astype(np.float32)
    centers = torch.from_numpy(c).cuda()
    f2cgt_amd.load().kmeans_slices_fit(torch.from_numpy(x).cuda(), None, centers, metric, 0, 0.0, 1.0, 1, 8)
    got = centers.cpu().numpy().astype(np.float64)
    for s in range(2):
        want = step64(x[s], np.ones(700, bool), c[s], metric)
        # a mean of fp64 sums rounded once per set and a few times behind them: below 2^-20 of the largest member
        assert (np.abs(got[s] - want) <= 1e-6 * np.abs(x[s]).max()).all()
        assert (np.abs(got[s] - want) <= 1e-6 * np.maximum(np.abs(want).max(1, keepdims=True), 8.0)).all()


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("value", [0.0, 1e-25, float("nan"), float("inf")])
def test_rows_left_out_do_not_count(metric, value):
    """Rows outside the mask that tie with every centre, or are no numbers: as if they were not there."""
    rng = np.random.default_rng(9)
    x, c = rng.standard_normal((3, 1000, 12)).astype(np.float32), rng.standard_normal((3, 50, 12)).astype(np.float32)
    keep = rng.random((3, 1000)) < 0.6
    x[~keep] = value
    padded = np.zeros((3, 1024), bool)
    padded[:, :1000] = keep
    bits = torch.from_numpy(np.packbits(padded, axis=1, bitorder="little").view(np.int32).copy()).cuda()
    centers = torch.from_numpy(c).cuda()
    f2cgt_amd.load().kmeans_slices_fit(torch.from_numpy(x).cuda(), bits, centers, metric, 0, 0.0, 1.0, 1, 8)
    got = centers.cpu().numpy().astype(np.float64)
    for s in range(3):
        mine = x[s][keep[s]]
        want = step64(mine, np.ones(len(mine), bool), c[s], metric)
        # fp64 sums, rounded once per set of rows: a few 2^-24 of the largest value
        assert np.abs(got[s] - want).max() <= 2.0 ** -21 * np.abs(mine).max()


def test_slices_stop_one_by_one():
    """A slice that has met the rule keeps its centres while the others go on; NaN in one flags only that one."""
    rng = np.random.default_rng(5)
    x = torch.from_numpy(rng.standard_normal((3, 2000, 8)).astype(np.float32)).cuda()
    x[1] = x[1, :1]                               # one point: final after the first step
    lib = f2cgt_amd.load()
    start = x[:, :16].clone() + 0.1
    once, more = start.clone(), start.clone()
    lib.kmeans_slices_fit(x, None, once, "l2", 2, 1e-9, 1.0, 2, 8)
    flags = lib.kmeans_slices_fit(x, None, more, "l2", 2, 1e-9, 1.0, 9, 3)
    assert flags.tolist()[1] == 1 and torch.equal(once[1], more[1]) and not torch.equal(once[0], more[0])
    x[2, 7, 3] = float("inf")
    assert lib.kmeans_slices_fit(x, None, start.clone(), "l2", 2, 1e-9, 1.0, 4, 8).tolist()[2] == 2


@pytest.mark.parametrize("m,n,k,rule", [(500, 40, 12, 2), (20000, 256, 16, 2), (500, 5, 3, 1), (3000, 130, 8, 0)])
def test_a_slice_without_rows_is_flagged(m, n, k, rule):
    """Its centres stay as they are; a slice with a single row that does not move its centre is no such slice."""
    g = torch.Generator().manual_seed(m)
    x, centers = torch.randn((3, m, k), generator=g).cuda(), torch.randn((3, n, k), generator=g).cuda()
    keep = torch.full((3, (m + 31) // 32), -1, dtype=torch.int32)
    keep[1] = 0
    keep[2] = 0
    keep[2, 3] = 1 << 5
    centers[2, n - 1] = x[2, 3 * 32 + 5]
    start = centers.clone()
    flags = f2cgt_amd.load().kmeans_slices_fit(x, keep.cuda(), centers, "l2", rule, 1e-9, 1.0, 1, 8)
    assert flags.tolist() == [0, 3, 0 if rule == 0 else 1]
    assert torch.equal(centers[1:], start[1:]) and not torch.equal(centers[0], start[0])


@pytest.mark.parametrize("dim,k,n", [(40, 16, 64), (33, 8, 32), (21, 7, 20), (16, 16, 256), (5, 8, 8)])
@pytest.mark.parametrize("where", ["device", "host", "double"])
def test_vq_metadata_as_slice_by_slice(dim, k, n, where, monkeypatch):
    """The same draws, the same rows, one step: the same codebooks to the rounding of the sums."""
    print("case vq_metadata", dim, k, n, where, flush=True)
    g = torch.Generator().manual_seed(dim)
    x = torch.randn((3000, dim), generator=g)
    x = x.cuda() if where == "device" else x.double() if where == "double" else x
    rows = torch.randperm(3000, generator=g)[:2500]
    torch.manual_seed(1)
    got = pipeline.vq_metadata(x, n, k, sample_index=rows, max_iter=1)
    after = torch.rand(1)
    monkeypatch.setattr(pipeline, "_train_all_slices", lambda *a: None)
    torch.manual_seed(1)
    want = pipeline.vq_metadata(x, n, k, sample_index=rows, max_iter=1)
    assert torch.equal(after, torch.rand(1)) and got.shape == want.shape
    assert torch.allclose(got, want, rtol=0, atol=2e-5)


def test_vq_metadata_refuses_ids_outside():
    x = torch.randn((500, 16), device="cuda")
    with pytest.raises(IndexError):
        pipeline.vq_metadata(x, 8, 8, sample_index=torch.tensor([1, 2, 500]))


@pytest.mark.parametrize("where", ["device", "host"])
@pytest.mark.parametrize("value,columns", [(float("nan"), 1), (float("inf"), 40), (1e30, 40)])
def test_vq_metadata_refuses_lengths_without_a_quantile(value, columns, where):
    """A NaN among a slice's lengths, or infinite lengths all over, keep no row: an error, not the random start."""
    x = torch.randn((500, 40), generator=torch.Generator().manual_seed(2))
    x[7 if columns == 1 else slice(None), -columns:] = value
    with pytest.raises(RuntimeError):
        pipeline.vq_metadata(x.cuda() if where == "device" else x, 8, 16, sample_index=torch.arange(400))


@pytest.mark.parametrize("where", ["device", "host"])
def test_vq_metadata_without_room_for_the_sample(where):
    """The sample of all slices does not fit: slice by slice, with the same draws."""
    x = torch.randn((60_000, 512), generator=torch.Generator().manual_seed(1))
    x = x.cuda() if where == "device" else x
    rows = torch.arange(0, 60_000)

    def train():
        torch.manual_seed(3)
        return pipeline.vq_metadata(x, 16, 16, sample_index=rows, max_iter=1)

    want = train()
    after = torch.rand(1)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info()[1]
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)    # the sample: 123 MB
    try:
        got = train()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(after, torch.rand(1))
    assert torch.allclose(got, want, rtol=0, atol=2e-5)
