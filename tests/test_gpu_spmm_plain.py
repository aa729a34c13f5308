"""spmm_csr on rows of uncompressed features: groups of lanes that hand the ids of a row round, at the edges of its batches
(8 source rows in flight, up to 64 ids a load) and of its widths.  The sums are in edge order, so results are bit-identical."""
import numpy as np
import pytest
import torch

import f2cgt_amd
import f2cgt_oracle as oc

pytestmark = pytest.mark.gpu


# groups of 8, 16, 32 and 64 lanes; lanes beyond the columns; two and three groups to a row; 4 k + 2 and odd columns
@pytest.mark.parametrize("dtype", [np.float32, np.float16, np.float64])
@pytest.mark.parametrize("dim", [8, 17, 20, 33, 64, 100, 128, 130, 260, 301, 602])
def test_rows_of_every_length(dtype, dim):
    rng = np.random.default_rng(dim)
    feat = rng.standard_normal((500, dim)).astype(dtype)
    deg = np.concatenate([[0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129, 0], rng.integers(0, 20, 300)])
    indptr = np.concatenate([[0], np.cumsum(deg)])
    indices = rng.integers(0, 500, indptr[-1])
    want = oc.spmm_csr(feat, indptr, indices)
    for index in (np.int32, np.int64):
        got = f2cgt_amd.load().spmm_csr(torch.from_numpy(feat).cuda(), torch.from_numpy(indptr.astype(index)).cuda(),
                                        torch.from_numpy(indices.astype(index)).cuda())
        assert np.array_equal(got.cpu().numpy(), want)


def test_more_rows_than_the_grid_has_groups():
    rows, dim = (1 << 15) * 8 + 37, 128                  # eight groups of 32 lanes to a workgroup, 2^15 row blocks
    feat = torch.randn((64, dim), device="cuda")
    indptr = torch.arange(rows + 1, device="cuda")
    indices = torch.randint(0, 64, (rows,), device="cuda")
    assert torch.equal(f2cgt_amd.load().spmm_csr(feat, indptr, indices), feat[indices])


# the same three times over: rows of three edges, which the groups that hand the ids round take
def test_more_rows_of_three_edges_than_the_grid_has_groups():
    rows, dim = (1 << 15) * 8 + 37, 128
    feat = 3.0 * torch.randint(-1000, 1000, (64, dim), device="cuda")          # exact sums and means
    indptr = torch.arange(0, 3 * rows + 1, 3, device="cuda")
    a = torch.randint(0, 64, (rows, 3), device="cuda")
    got = f2cgt_amd.load().spmm_csr(feat, indptr, a.flatten())
    assert torch.equal(got, (feat[a[:, 0]] + feat[a[:, 1]] + feat[a[:, 2]]) / 3)


def test_infinities_and_nans_stay_in_their_rows():
    feat = torch.zeros((4, 100), device="cuda")
    feat[1, 3], feat[2, 4] = float("inf"), float("nan")
    got = f2cgt_amd.load().spmm_csr(feat, torch.tensor([0, 2, 2, 4], device="cuda"), torch.tensor([0, 1, 3, 2], device="cuda"))
    assert torch.isinf(got[0, 3]) and torch.isnan(got[2, 4])
    assert int((got != 0).sum()) == 2
    got = f2cgt_amd.load().spmm_csr(feat, torch.tensor([0, 4, 4, 9], device="cuda"),
                                    torch.tensor([0, 1, 0, 0, 3, 2, 0, 3, 0], device="cuda"))   # three edges per row and more
    assert torch.isinf(got[0, 3]) and torch.isnan(got[2, 4])
    assert int((got != 0).sum()) == 2
