"""Row offsets that decrease: sums of the rows concerned are wrong, nothing is read outside the operands, and blocks of rows
with ordinary offsets keep their results."""
import numpy as np
import pytest
import torch

import f2cgt_oracle as oc
from f2cgt_amd import capi

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def graph(rng, rows, fanout, n):
    """Rows of `fanout` edges; in 64 rows in the middle two offsets of every eight are replaced by one far ahead and one
    behind.  -> indptr, indices, the rows at least 256 (the largest block) away from a replaced offset."""
    indptr = np.arange(rows + 1, dtype=np.int64) * fanout
    lo = rows // 2 // 64 * 64
    for r in range(lo, lo + 64, 8):
        indptr[r + 2] = min(indptr[r + 2] + 40 * fanout, rows * fanout)
        indptr[r + 5] = max(indptr[r + 5] - 40 * fanout, 0)
    sound = np.ones(rows, dtype=bool)
    sound[max(0, lo - 256):lo + 320] = False
    return indptr, rng.integers(0, n, size=rows * fanout), sound


@pytest.mark.parametrize("idx", [np.int64, np.int32])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
@pytest.mark.parametrize("books", [1, 3])
def test_log_sq_with_decreasing_offsets(bits, books, idx):
    rng = np.random.default_rng(bits + 10 * books)
    n = 3000
    cb = np.repeat(np.array([[0.01, 3.0, -6.643856, 1.5849625, 0.4]], dtype=np.float32), books, axis=0)
    for feat_dim in (64, 66, 300, 602):
        column_slice = (-(-feat_dim // books) + 7) // 8 * 8
        codes = rng.integers(0, 256, size=(n, (feat_dim * bits + 7) // 8), dtype=np.uint8)
        stored = codes.view(np.int8) if bits == 8 else codes
        for rows, fanout in ((900, 1), (900, 10), (600, 40), (700, 300)):
            print("case log sq bits=%d books=%d dim=%d rows=%d fanout=%d" % (bits, books, feat_dim, rows, fanout), flush=True)
            indptr, indices, sound = graph(rng, rows, fanout, n)
            got = capi.sq_decompress_spmm_csr(dev(stored), dev(cb), dev(indptr.astype(idx)), dev(indices.astype(idx)), bits,
                                              column_slice, feat_dim)
            torch.cuda.synchronize()
            plain = np.arange(rows + 1, dtype=np.int64) * fanout
            want = oc.sq_decompress_spmm_csr(stored, cb, plain, indices, bits, column_slice, feat_dim)
            assert sound.any() and np.allclose(got.cpu().numpy()[sound], want[sound], rtol=1e-5, atol=3e-5)


@pytest.mark.parametrize("idx", [np.int64, np.int32])
@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_affine_sq_with_decreasing_offsets(bits, idx):
    rng = np.random.default_rng(bits)
    n = 3000
    for feat_dim in (64, 66, 300, 602):
        codes = rng.integers(0, 256, size=(n, (feat_dim * bits + 7) // 8), dtype=np.uint8)
        params = np.stack([rng.standard_normal(feat_dim) - 3, 0.01 + 0.02 * rng.random(feat_dim)]).astype(np.float32)
        for rows, fanout in ((900, 1), (900, 10), (600, 40), (700, 300)):
            print("case affine sq bits=%d dim=%d rows=%d fanout=%d" % (bits, feat_dim, rows, fanout), flush=True)
            indptr, indices, sound = graph(rng, rows, fanout, n)
            got = capi.sq_affine_decompress_spmm_csr(dev(codes), dev(params), dev(indptr.astype(idx)),
                                                     dev(indices.astype(idx)), bits, feat_dim)
            torch.cuda.synchronize()
            plain = np.arange(rows + 1, dtype=np.int64) * fanout
            want = oc.sq_affine_decompress_spmm_csr(codes, params, plain, indices, bits, feat_dim)
            assert np.allclose(got.cpu().numpy()[sound], want[sound], rtol=1e-5, atol=1e-5 * np.abs(want).max())


@pytest.mark.parametrize("idx", [np.int64, np.int32])
def test_hybrid_with_decreasing_offsets(idx):
    rng = np.random.default_rng(4)
    n, n_sq, w = 3000, 1200, 16
    row_map = np.empty(n, dtype=np.int32)
    row_map[:n_sq] = rng.permutation(n_sq)
    row_map[n_sq:] = -rng.permutation(n - n_sq) - 1
    for feat_dim in (48, 128):
        sq_codes = rng.integers(0, 256, size=(n_sq, feat_dim), dtype=np.uint8)
        params = np.stack([rng.standard_normal(feat_dim) - 3, 0.01 + 0.02 * rng.random(feat_dim)]).astype(np.float32)
        vq_codes = rng.integers(0, 256, size=(n - n_sq, feat_dim // w), dtype=np.uint8)
        vcb = rng.standard_normal((feat_dim // w, 256, w)).astype(np.float32)
        for rows, fanout in ((900, 1), (900, 10), (600, 40), (700, 300)):
            print("case hybrid dim=%d rows=%d fanout=%d" % (feat_dim, rows, fanout), flush=True)
            indptr, indices, sound = graph(rng, rows, fanout, n)
            got = capi.hybrid_decompress_spmm_csr(dev(row_map), dev(sq_codes), dev(params), dev(vq_codes), dev(vcb),
                                                  dev(indptr.astype(idx)), dev(indices.astype(idx)), feat_dim)
            torch.cuda.synchronize()
            plain = np.arange(rows + 1, dtype=np.int64) * fanout
            want = oc.hybrid_decompress_spmm_csr(row_map, sq_codes, params, vq_codes, vcb, plain, indices, feat_dim)
            assert np.allclose(got.cpu().numpy()[sound], want[sound], rtol=1e-5, atol=8e-5)
