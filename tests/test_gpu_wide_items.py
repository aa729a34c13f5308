"""Log-domain rows with one codebook whose codes are read where they are: items of eight columns, or of four in short
launches of 8-bit rows.  The same values in the same order as decoding the rows and aggregating them, so bit for bit the same."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    from f2cgt_amd import capi, synth

pytestmark = pytest.mark.gpu

# widths about whole items and, for 2 and 4 bits, about the line between staged (four columns) and direct
WIDTHS = [(8, d) for d in (8, 10, 12, 14, 16, 18, 130, 254, 602, 1030)] + \
         [(4, d) for d in (16, 254, 256, 258, 260, 262, 264, 602)] + [(2, d) for d in (32, 512, 514, 516, 518, 520, 1030)]


def test_eight_bit_rows_on_both_sides_of_a_short_launch():
    for dim in (8, 10, 12, 14, 20, 66, 126, 128, 130, 132):
        for rows in (16384, 16385):
            test_equal_to_decode_and_aggregate(8, dim, rows, 6)


@pytest.mark.parametrize("bits,dim", WIDTHS)
@pytest.mark.parametrize("rows,longest", [(1, 5), (7, 20), (300, 20), (2050, 6), (40, 900)])
def test_equal_to_decode_and_aggregate(bits, dim, rows, longest):
    g = torch.Generator(device="cuda")
    g.manual_seed(dim * 1000 + rows + bits)
    n, row = 501, (dim * bits + 7) // 8
    # the table ends with its last row: what is read behind it would not be the table's
    codes = torch.randint(-128, 128, (n, row), generator=g, device="cuda", dtype=torch.int8)
    book = torch.tensor([[0.006, 2.8, -7.38, 1.485, 0.8123]], device="cuda")
    width = (dim + 7) // 8 * 8
    decoded = capi.sq_decompress(codes, book, bits, width, dim)
    deg = torch.randint(0, longest + 1, (rows,), generator=g, device="cuda")
    deg[0] = longest
    for dtype, mode in ((torch.int64, capi.STORE_STREAM), (torch.int32, capi.STORE_CACHED)):
        indptr = synth.csc_from_degrees(deg, dtype)
        indices = torch.randint(0, n, (int(indptr[-1]),), generator=g, device="cuda").to(dtype)
        indices[-1] = n - 1
        want = capi.spmm_csr(decoded, indptr, indices)
        room = torch.full((rows + 8, dim), 5.0, device="cuda")      # four guard rows on either side
        was = capi.set_store_mode(mode)
        try:
            capi.sq_decompress_spmm_csr(codes, book, indptr, indices, bits, width, dim, out=room[4:rows + 4])
        finally:
            capi.set_store_mode(was)
        assert torch.equal(room[4:rows + 4], want)
        assert bool((room[:4] == 5.0).all()) and bool((room[rows + 4:] == 5.0).all())
