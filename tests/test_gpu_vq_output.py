"""The fused VQ kernel's output, written by lane swaps and with stores beyond the columns dropped: partial column tiles, a
last pass of one to three rows, one to four lane groups per row, nothing touched around the result."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    from f2cgt_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,w", [(16, 8), (64, 8), (72, 8), (120, 8), (128, 32), (136, 8), (192, 32), (264, 8), (602, 32), (130, 16),
                                   (100, 8)])
@pytest.mark.parametrize("fanout", [3, 12, 24, 50])
@pytest.mark.parametrize("codes_per_book", [256, 17])
def test_rows_and_columns_at_the_edges_of_tiles(dim, w, fanout, codes_per_book):
    g = torch.Generator(device="cuda")
    g.manual_seed(dim * 64 + fanout)
    books, n = -(-dim // w), 3001
    codes = torch.randint(0, codes_per_book, (n, books), generator=g, device="cuda", dtype=torch.uint8)
    cbs = torch.randn((books, codes_per_book, w), generator=g, device="cuda")
    decoded = torch.cat([cbs[i][codes[:, i].long()] for i in range(books)], 1)[:, :dim].double()
    for rows in (256, 257, 258, 259, 12 * 1024 + 5):
        deg = torch.full((rows,), fanout, device="cuda") if rows % 2 else torch.randint(0, 2 * fanout, (rows,), generator=g,
                                                                                        device="cuda")
        indptr = synth.csc_from_degrees(deg, torch.int64)
        indices = torch.randint(0, n, (int(indptr[-1]),), generator=g, device="cuda")
        room = torch.full((rows + 8, dim), 5.0, device="cuda")     # four guard rows on either side (16-byte aligned)
        capi.vq_decompress_spmm_csr(codes, cbs, indptr, indices, dim, out=room[4:rows + 4])
        assert bool((room[:4] == 5.0).all()) and bool((room[rows + 4:] == 5.0).all())
        got = room[4:rows + 4]
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"), deg)
        want = torch.zeros((rows, dim), dtype=torch.float64, device="cuda").index_add_(0, row, decoded[indices])
        want /= deg.clamp(min=1).double()[:, None]
        # n - 1 additions of values up to max|x| in any order, each rounded by half a unit of a sum of at most n max|x|,
        # over n, and a mean within two units
        bound = (deg.clamp(min=1).double()[:, None] + 4.0) * 2.0 ** -24 * float(decoded.abs().max())
        assert bool(((got.double() - want).abs() <= bound).all()), rows
        one = deg == 1
        assert torch.equal(got[one].double(), want[one])
