"""Codes of a whole table in one launch (f2cgt_vq_encode_slices) against the oracle's labels of every column slice."""
import numpy as np
import pytest
import torch

import f2cgt_oracle as oc
import f2cgt_amd
from f2cgt_amd import capi, pipeline

pytestmark = pytest.mark.gpu


def padded(table, s, k):
    part = table[:, s * k:(s + 1) * k]
    return np.ascontiguousarray(np.pad(part, ((0, 0), (0, k - part.shape[1]))))


# m: below, at and beyond a wave's 64 rows, and more shares than rows; dim: a last slice of 1 to k columns, fewer than eight
# columns in all, one slice; start / pitch: rows that begin at any float and leave a gap; n: one padded tile, all of it used
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("m,dim,k,n,start,pitch", [
    (1, 3, 8, 5, 0, 3), (63, 16, 16, 32, 0, 16), (64, 100, 16, 256, 0, 100), (65, 33, 32, 33, 1, 37), (3000, 137, 32, 256, 3, 141),
    (700, 96, 8, 200, 2, 99), (129, 40, 24, 256, 1, 41), (2500, 90, 48, 256, 0, 90), (500, 130, 64, 64, 1, 131), (70, 600, 8, 16, 0, 600),
    (200, 17, 32, 7, 5, 23)])
def test_vq_encode_slices(metric, m, dim, k, n, start, pitch):
    print("case vq_encode_slices", metric, m, dim, k, n, start, pitch, flush=True)
    rng = np.random.default_rng(m + dim + k)
    slices = (dim + k - 1) // k
    table = rng.standard_normal((m, dim)).astype(np.float32)
    books = rng.standard_normal((slices, n, k)).astype(np.float32)           # nonzero also beyond the table's last column
    flat = torch.zeros(m * pitch + start, device="cuda")
    x = flat[start:].view(m, pitch)[:, :dim]
    x.copy_(torch.from_numpy(table))
    out = torch.full((m + 2, slices + 3), 77, dtype=torch.uint8, device="cuda")
    assert f2cgt_amd.load().vq_encode_slices(x, torch.from_numpy(books).cuda(), out[1:m + 1, 1:slices + 1], metric)
    got = out.cpu().numpy()
    for s in range(slices):
        want, near = oc.kmeans_predict(padded(table, s, k), books[s], metric)
        assert np.array_equal(got[1:m + 1, 1 + s][~near], want[~near]) and near.mean() < 0.02
    got[1:m + 1, 1:slices + 1] = 77
    assert (got == 77).all()                                                 # nothing else is written


def test_vq_encode_slices_leaves_other_calls():
    lib = f2cgt_amd.load()
    x, books = torch.randn((10, 20), device="cuda"), torch.randn((2, 16, 10), device="cuda")
    out = torch.empty((10, 2), dtype=torch.uint8, device="cuda")
    assert lib.vq_encode_slices(x, books, out, "cosine")
    assert not lib.vq_encode_slices(x.double(), books, out, "cosine")
    assert not lib.vq_encode_slices(x.t().contiguous().t(), books, out, "cosine")
    assert not lib.vq_encode_slices(x, torch.randn((2, 300, 10), device="cuda"), out, "cosine")
    assert not lib.vq_encode_slices(x, torch.randn((2, 16, 20), device="cuda"), out, "cosine")      # a slice without columns
    assert not lib.vq_encode_slices(x[:1].expand(10, 20), books, out, "cosine")


@pytest.mark.parametrize("dim,k,n", [(100, 16, 256), (45, 8, 40), (70, 70, 16)])
def test_vq_compress_equals_its_slices(dim, k, n):
    """One launch, the same rows from the host (slice by slice), and rows that are not contiguous: the same codes."""
    rng = np.random.default_rng(dim)
    x = torch.from_numpy(rng.standard_normal((1000, dim)).astype(np.float32))
    books = torch.from_numpy(rng.standard_normal(((dim + k - 1) // k, n, k)).astype(np.float32)).cuda()
    by_slice, _ = pipeline.vq_compress(x, n, k, codebooks=books)
    for features in (x.cuda(), x.cuda().t().contiguous().t()):
        codes, _ = pipeline.vq_compress(features, n, k, codebooks=books, batch_rows=600)
        assert torch.equal(codes, by_slice)


@pytest.mark.parametrize("metric", ["l2", "cosine"])
@pytest.mark.parametrize("n,k", [(2, 3), (2, 4), (34, 8), (100, 13), (256, 16), (254, 16), (256, 17)])
def test_kmeans_predict_close_pairs(metric, n, k):
    """Centres in pairs 2^-10 to 2^-15 of their size apart: from 4 to 16 dimensions the lowest four bits of a score are its slot,
    which changes scores by as much as what tells the two of a pair apart, and some of the slots are padding."""
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((4000, k)).astype(np.float32)
    c = rng.standard_normal((n, k)).astype(np.float32)
    c[1::2] = c[0::2] * (1 + rng.choice([-1, 1], (n // 2, k)) * 2.0 ** -rng.integers(10, 16, (n // 2, 1))).astype(np.float32)
    want, near = oc.kmeans_predict(x, c, metric)
    got = capi.kmeans_predict(torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda(), metric).cpu().numpy()
    # a cosine gap is about 2^-j / sqrt(k) wide, the oracle's near-ties are those below 1e-6: 7 % of the rows of one pair in
    # 4 dimensions, 1 to 3 % where the rows spread over many pairs
    assert near.mean() < 0.1 and np.array_equal(got[~near], want[~near])


@pytest.mark.parametrize("n", [33, 256])
@pytest.mark.parametrize("k", [2, 4, 8, 16, 17])
def test_l2_scores_beyond_the_largest_float(n, k):
    """|x|^2 = 1e38 and |c|^2 = 2e38: |c|^2 - 2 x . c is infinite in fp32 for centres on the far side, |x|^2 + |c|^2 is not."""
    rng = np.random.default_rng(n + k)
    x, c = rng.standard_normal((3000, k)), rng.standard_normal((n, k))
    x = (x / np.linalg.norm(x, axis=1, keepdims=True) * 1e19).astype(np.float32)
    c = (c / np.linalg.norm(c, axis=1, keepdims=True) * 2 ** 0.5 * 1e19).astype(np.float32)
    want, near = oc.kmeans_predict(x, c, "l2")
    assert ((c[None].astype(np.float64) ** 2).sum(2) - 2 * x.astype(np.float64) @ c.T.astype(np.float64)).max() > 3.41e38
    got = capi.kmeans_predict(torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda(), "l2").cpu().numpy()
    assert near.mean() < 0.01 and np.array_equal(got[~near], want[~near])


@pytest.mark.parametrize("metric", ["l2", "cosine"])
@pytest.mark.parametrize("k", [4, 8, 16])
@pytest.mark.parametrize("what", ["one centre", "zero rows", "all zero", "nan centres", "only nan centres", "infinite centre"])
def test_scores_that_are_zero_or_no_numbers(what, k, metric):
    """The same rows and centres with zeros up to 17 dimensions take plain scores: the same labels.  A zero score with a slot
    in its low bits is a denormal number; a centre that is no number is never nearest."""
    rng = np.random.default_rng(k)
    n = 1 if what == "one centre" else 70
    x, c = rng.standard_normal((1000, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    if what == "zero rows":
        x[::3], c[5] = 0, 0
    elif what == "all zero":
        x[:], c[:] = 0, 0
    elif what == "nan centres":
        c[::7, 1] = np.nan
    elif what == "only nan centres":
        c[:] = np.nan
    elif what == "infinite centre":
        c[9, 0] = np.inf

    def labels(k_pad):
        pad = [torch.from_numpy(np.pad(a, ((0, 0), (0, k_pad - k)))).cuda() for a in (x, c)]
        return capi.kmeans_predict(*pad, metric).cpu().numpy()

    got = labels(k)
    assert got.min() >= 0 and got.max() < n and np.array_equal(got, labels(17))
    if metric == "cosine" and what == "nan centres":
        assert not np.isin(got, np.arange(0, n, 7)).any()
    if what in ("one centre", "all zero", "only nan centres"):
        assert not got.any()
