"""Order statistics of |x| per column slice (f2cgt_abs_order_stats) against a sorted copy, and the SQ codebooks made from
them against numpy's percentiles."""
import numpy as np
import pytest
import torch

import f2cgt_amd
import f2cgt_oracle as oc

pytestmark = pytest.mark.gpu


def _values(kind, rng, n, d):
    if kind == "normal":
        return rng.standard_normal((n, d)).astype(np.float32) * np.float32(3)
    if kind == "equal":
        return np.full((n, d), -0.75, dtype=np.float32)
    if kind == "bits":         # every exponent, denormal numbers and infinities among them
        bits = rng.integers(0, 0x7f800001, size=(n, d), dtype=np.uint32) | (rng.integers(0, 2, size=(n, d), dtype=np.uint32) << 31)
        return bits.view(np.float32)
    return np.where(rng.random((n, d)) < 0.6, 0.0, rng.standard_normal((n, d))).astype(np.float32)   # mostly zeros


# one value; a row wider than a workgroup; slices of 8 with a ragged last one; odd widths (scalar loads), pairs, quads;
# more slices than workgroups per slice; enough rows for every workgroup and an odd remainder
@pytest.mark.parametrize("kind", ["normal", "equal", "bits", "sparse"])
@pytest.mark.parametrize("n,d,slice_", [(1, 1, 1), (3, 1500, 1500), (4097, 20, 8), (5000, 7, 7), (2049, 30, 30),
                                        (700, 602, 8), (40001, 100, 104), (1023, 4100, 4100),
                                        # what a wave hands from the second pass to the third: one value less than fits,
                                        # exactly that many, one more; more workgroups than hand anything on
                                        (8191, 1, 1), (8192, 1, 1), (8193, 1, 1), (300, 2100, 2), (300, 2100, 8)])
def test_ranks_sum_and_flag(kind, n, d, slice_):
    rng = np.random.default_rng(n + d)
    table = _values(kind, rng, n + 50, d)
    rows = rng.integers(-n, n + 50, size=n)
    sample = np.abs(table[rows])
    count = (d + slice_ - 1) // slice_
    widths = [min(slice_, d), d - (count - 1) * slice_]
    ranks = []
    for w in widths:
        total = n * w
        ranks += [0, total // 200, total * 199 // 200, total - 1]
    got = f2cgt_amd.load().abs_order_stats(torch.from_numpy(table).cuda(), torch.from_numpy(rows).cuda(), slice_, ranks)
    got = got.cpu().numpy()
    assert got.shape == (count, 6)
    for i in range(count):
        part = np.sort(sample[:, i * slice_:(i + 1) * slice_].ravel())
        want = part[ranks[4:] if i == count - 1 else ranks[:4]]
        assert np.array_equal(got[i, :4].astype(np.float32), want)
        assert got[i, 5] == 0.0
        # fp64 sums of non-negative values in any order: (number of terms) roundings of the total at most
        assert np.allclose(got[i, 4], part.sum(dtype=np.float64), rtol=part.size * 2.0 ** -52)


def test_a_nan_is_reported():
    x = torch.rand((3000, 24), device="cuda")
    x[2111, 17] = float("nan")
    got = f2cgt_amd.load().abs_order_stats(x, None, 8, [0, 1, 2, 3] * 2).cpu()
    assert got[:, 5].tolist() == [0.0, 0.0, 1.0]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n,d,slice_", [(2000, 100, 104), (1501, 37, 16)])
def test_codebooks_on_the_device_are_numpys(dtype, n, d, slice_):
    from f2cgt_amd import pipeline
    rng = np.random.default_rng(d)
    x = torch.from_numpy(rng.standard_normal((n, d)).astype(np.float32)).to(dtype)
    pick = torch.from_numpy(rng.permutation(n)[:n * 3 // 4])
    for where in ("cuda", "cpu"):
        _, books = pipeline.sq_compress(x.to(where), 4, slice_, sample_index=pick)
        for i in range(books.shape[0]):
            want = oc.sq_codebook(x[pick].float().numpy()[:, i * slice_:(i + 1) * slice_])
            got = books[i].cpu().numpy()
            assert np.array_equal(got[:4], want[:4]) and np.isclose(got[4], want[4], rtol=1e-6)
    one = np.array([float(v) for v in pipeline.sq_metadata(x[pick].cuda())], dtype=np.float32)
    want = oc.sq_codebook(x[pick].float().numpy())
    assert np.array_equal(one[:4], want[:4]) and np.isclose(one[4], want[4], rtol=1e-6)


@pytest.mark.parametrize("where", ["cuda", "cpu"])
@pytest.mark.parametrize("bad", [300, -301, 2 ** 40])
def test_sample_ids_outside_the_table_are_refused(where, bad):
    from f2cgt_amd import pipeline
    x = torch.rand((300, 24))
    pick = torch.arange(-300, 300)
    if where == "cuda":      # on the host the same list is refused by the gather
        got = f2cgt_amd.load().abs_order_stats(x.cuda(), pick.cuda(), 8, [0, 1, 2, 3] * 2).cpu()
        assert got[:, 5].tolist() == [0.0, 0.0, 0.0]
    pick[77] = bad
    with pytest.raises(IndexError):
        pipeline.sq_compress(x.to(where), 4, 8, sample_index=pick)


def test_rows_that_overlap():
    """A row expanded to a table (row stride 0) and a one-row table seen through a transpose (row stride 1)."""
    from f2cgt_amd import pipeline
    row = torch.randn((1, 40), generator=torch.Generator().manual_seed(3))
    pick = torch.arange(0, 300, 3)
    for table, rows in ((row.cuda().expand(300, 40), pick), (torch.randn((40, 1)).cuda().t(), torch.zeros(5, dtype=torch.int64))):
        assert table.stride(0) < table.shape[1]
        whole = torch.empty(table.shape, device="cuda").copy_(table)
        codes, books = pipeline.sq_compress(table, 4, 16, sample_index=rows)
        want_codes, want_books = pipeline.sq_compress(whole, 4, 16, sample_index=rows)
        assert torch.equal(books, want_books) and torch.equal(codes, want_codes)
        assert [float(v) for v in pipeline.sq_metadata(table)] == [float(v) for v in pipeline.sq_metadata(whole)]


@pytest.mark.parametrize("kind", ["columns apart", "one row expanded"])
def test_a_table_that_is_no_plain_one_is_not_copied_whole(kind):
    from f2cgt_amd import pipeline
    table = torch.randn((40, 100000), device="cuda").t() if kind == "columns apart" else torch.randn((1, 40), device="cuda").expand(100000, 40)
    pick = torch.arange(0, 100000, 100)
    _, want = pipeline.sq_compress(table[pick.cuda()], 4, 16, sample_index=torch.arange(1000))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    codes, books = pipeline.sq_compress(table, 4, 16, sample_index=pick, batch_rows=1000)
    assert torch.equal(books, want)
    # the codes, the sample and scratch of a few MB; the table is 16 MB
    assert torch.cuda.max_memory_allocated() - before - codes.numel() < 12 << 20


@pytest.mark.parametrize("where", ["cuda", "cpu"])
def test_samples_of_any_shape(where, monkeypatch):
    """A list of lists of ids, a single id, a mask; a host sample that the GPU has no room for; more values than the
    device counts (the limit lowered): the codebooks of the flat list, and numpy's, as from a host table."""
    from f2cgt_amd import pipeline
    rng = np.random.default_rng(9)
    x = torch.from_numpy(rng.standard_normal((400, 30)).astype(np.float32))
    pick = torch.from_numpy(rng.permutation(400)[:240])
    table = x.to(where)

    def books(index):
        return pipeline.sq_compress(table, 4, 8, sample_index=index)[1].cpu().numpy()

    want = np.stack([oc.sq_codebook(x[pick].numpy()[:, lo:lo + 8]) for lo in range(0, 30, 8)])
    mask = torch.zeros(400, dtype=torch.bool)
    mask[pick] = True
    for index in (pick, pick.view(12, 20), pick.int(), mask):
        got = books(index)
        assert np.array_equal(got[:, :4], want[:, :4]) and np.allclose(got[:, 4], want[:, 4], rtol=1e-6)
    one = np.stack([oc.sq_codebook(x[7].numpy()[None, lo:lo + 8]) for lo in range(0, 30, 8)])
    assert np.array_equal(books(torch.tensor(7))[:, :4], one[:, :4])
    whole = [float(v) for v in pipeline.sq_metadata(table)]
    assert [float(v) for v in pipeline.sq_metadata(table.view(20, 20, 30))] == whole
    assert float(pipeline.sq_metadata(table[3, 3])[0]) == max(abs(float(x[3, 3])), 1e-5)

    monkeypatch.setattr(pipeline, "_device_takes", lambda *sizes: False)
    monkeypatch.setattr(pipeline, "_device_statistics", None)
    assert np.array_equal(books(pick)[:, :4], want[:, :4])
    monkeypatch.undo()

    def full(*args, **kwargs):
        raise torch.OutOfMemoryError("no room")
    if where == "cpu":
        with monkeypatch.context() as m:
            to_gpu = torch.Tensor.cuda
            m.setattr(torch.Tensor, "cuda", lambda t, *a, **k: full() if t.shape in ((240, 30), (240, 8)) else to_gpu(t, *a, **k))
            assert np.array_equal(books(pick)[:, :4], want[:, :4])


def test_features_that_require_a_gradient_are_refused():
    from f2cgt_amd import pipeline
    table = torch.randn((300, 24), device="cuda", requires_grad=True)
    pick = torch.arange(0, 300, 2)
    for call in (lambda: pipeline.sq_compress(table, 4, 8, sample_index=pick), lambda: pipeline.sq_metadata(table)):
        with pytest.raises(RuntimeError, match="requires grad"):
            call()
    with torch.no_grad():
        assert torch.equal(pipeline.sq_compress(table, 4, 8, sample_index=pick)[1],
                           pipeline.sq_compress(table.detach(), 4, 8, sample_index=pick)[1])


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_row_ids_on_another_device_are_refused():
    with pytest.raises(RuntimeError, match="on the device of x"):
        f2cgt_amd.load().abs_order_stats(torch.rand((30, 8), device="cuda:0"), torch.arange(5, device="cuda:1"), 8, [0, 1, 2, 3] * 2)


# tables whose rows have a pitch and start at any float, as a column range of a wider table has them: quads, pairs and single
# floats per load, whole slices and a ragged last one; with a row list, and all rows without one
@pytest.mark.parametrize("listed", [True, False])
@pytest.mark.parametrize("n,d,slice_,start,pitch", [(3001, 32, 16, 4, 40), (3001, 32, 16, 2, 42), (3001, 32, 16, 1, 40), (2000, 30, 8, 6, 36),
                                                    (2000, 31, 31, 3, 37), (40001, 100, 104, 4, 104), (70, 602, 602, 1, 605), (1, 24, 8, 5, 40)])
def test_rows_with_a_pitch(listed, n, d, slice_, start, pitch):
    rng = np.random.default_rng(n + start)
    wide = rng.standard_normal((n, pitch)).astype(np.float32)
    wide[:, :start] = wide[:, start + d:] = 1e30                     # what lies between the rows must not be counted
    table = torch.from_numpy(wide).cuda()[:, start:start + d]
    rows = rng.integers(-n, n, size=n // 2 + 1) if listed else np.arange(n)
    m, count = rows.size, (d + slice_ - 1) // slice_
    ranks = []
    for w in (min(slice_, d), d - (count - 1) * slice_):
        ranks += [0, m * w // 3, m * w * 2 // 3, m * w - 1]
    got = f2cgt_amd.load().abs_order_stats(table, torch.from_numpy(rows).cuda() if listed else None, slice_, ranks).cpu().numpy()
    sample = np.abs(wide[:, start:start + d][rows])
    for i in range(count):
        part = np.sort(sample[:, i * slice_:(i + 1) * slice_].ravel())
        assert np.array_equal(got[i, :4].astype(np.float32), part[ranks[4:] if i == count - 1 else ranks[:4]]) and got[i, 5] == 0.0
        assert np.allclose(got[i, 4], part.sum(dtype=np.float64), rtol=part.size * 2.0 ** -52)


@pytest.mark.parametrize("scale", [1e-7, 1e-3, 1.0, 1e6])
@pytest.mark.parametrize("n,d,slice_", [(1, 1, 8), (3, 5, 2), (2000, 33, 16), (300, 64, 64)])
def test_codebooks_made_on_the_device(n, d, slice_, scale):
    """Percentiles, floors and the lifted mean as from the statistics on the host; log2 correctly rounded."""
    from f2cgt_amd import pipeline
    x = (torch.randn((n, d), generator=torch.Generator().manual_seed(n + d)) * scale).cuda()
    places = pipeline._percentile_places(n, d, slice_)[1]
    books, stats = f2cgt_amd.load().sq_codebooks(x, None, slice_, [r for s in places for p in s for r in p[:2]],
                                                 [p[2] for s in places for p in s])
    want = [[float(v) for v in pipeline._sq_codebook(*values)] for values in pipeline._device_statistics(x, None, slice_)]
    got, want = books.cpu().numpy(), np.array(want, dtype=np.float32)
    assert np.array_equal(got[:, [0, 1, 4]], want[:, [0, 1, 4]]) and not stats.cpu()[:, 5].any()
    assert np.array_equal(got[:, 2], np.log2(got[:, 0].astype(np.float64)).astype(np.float32))
    assert np.array_equal(got[:, 3], np.log2(got[:, 1].astype(np.float64)).astype(np.float32) + np.float32(1e-5))


def test_codebook_of_a_nan():
    x = torch.rand((500, 16), device="cuda")
    x[3, 9] = float("nan")
    from f2cgt_amd import pipeline
    books = pipeline.sq_compress(x, 4, 8, sample_index=torch.arange(500))[1].cpu()
    assert not torch.isnan(books[0]).any() and torch.isnan(books[1]).all()
