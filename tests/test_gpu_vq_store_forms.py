"""The fused VQ operator with tables and outputs around the size of the last-level cache, and rows of split pieces, against
decode + spmm_csr."""
import pytest
import torch

import f2cgt_amd

pytestmark = pytest.mark.gpu


# rows of 600 and 680 columns and an output of 100 MB; 200 columns, an output beyond the last-level cache; a table beyond it
@pytest.mark.parametrize("n_src,books,width,dim,rows,fanout", [(3000, 19, 32, 600, 41_667, 12), (3000, 85, 8, 680, 36_765, 9),
                                                               (3000, 25, 8, 200, 335_545, 10), (16_777_217, 16, 8, 128, 65_537, 15),
                                                               (16_777_217, 25, 8, 200, 125_001, 12), (16_777_217, 27, 8, 216, 115_741, 13),
                                                               (16_777_217, 16, 8, 128, 122_881, 15), (16_777_217, 17, 16, 256, 61_441, 10),
                                                               (8_388_609, 33, 16, 512, 49_153, 11), (16_777_217, 25, 8, 200, 125_001, 13),
                                                               # large outputs of few edges per row: half a last tile, whole tiles
                                                               (3000, 12, 16, 192, 349_526, 3), (3000, 24, 8, 192, 349_527, 8),
                                                               (3000, 14, 32, 448, 149_799, 5), (3000, 11, 16, 176, 381_303, 6),
                                                               (3000, 24, 16, 384, 174_763, 3), (3000, 16, 16, 256, 262_145, 5)])
@pytest.mark.parametrize("ragged", [False, True])
def test_store_forms_agree_with_the_unfused_operators(n_src, books, width, dim, rows, fanout, ragged):
    capi = f2cgt_amd.load()
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    table = torch.randint(0, 256, (n_src, books), generator=g, device="cuda", dtype=torch.uint8)
    cb = torch.randn((books, 256, width), generator=g, device="cuda")
    deg = torch.full((rows,), fanout, device="cuda")
    if ragged:      # the same number of edges but one, row lengths from 0 to past a mini-block's staging
        deg = torch.randint(0, 2 * fanout, (rows,), generator=g, device="cuda")
        deg[rows // 2] = 150
    indptr = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(deg, 0)])
    used = torch.randint(0, n_src, (3000,), generator=g, device="cuda")
    pick = torch.randint(0, 3000, (int(indptr[-1]),), generator=g, device="cuda")
    got = capi.vq_decompress_spmm_csr(table, cb, indptr, used[pick], dim)
    decoded = capi.vq_decompress(table[used], cb, dim)
    want = capi.spmm_csr(decoded, indptr, pick)
    # two fp32 sums of the same n terms in any order, each with one rounding per addition and two for the mean
    bound = 2 * (deg.unsqueeze(1) + 2) * 2.0 ** -24 * capi.spmm_csr(decoded.abs(), indptr, pick)
    assert bool(((got - want).abs() <= bound).all())
